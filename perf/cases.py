"""The fused embedding path as users run it, as cases that can be timed and compared.

A case names one of the prebuilt libraries (``recflex_amd.prebuilt``: the benchmark's models C1-C5
with their tuned schedules or the default ones, the models shaped like the reference's own, the
skewed and the few-long-bags model) and what a caller varies without building again: the batch,
the rows of the tables, the length of the bags, and the entry point.

entry
    ``bound``   ``FeatEmbed.forward_indices(bound, out=...)``: inputs bound once, the serving loop
    ``lists``   ``FeatEmbed.forward_indices(indices, offsets)``: per-feature tensors on every call
    ``packed``  ``FeatEmbed.forward(arg_buffers, ...)``: the packed buffer of ``FeatPreprocess``
    ``model``   ``RecomModel.forward`` on the packed buffer: embedding, then the MLP of
                ``examples/end_to_end.py``
    ``text``    ``FeatProcessEmbed.forward(raw_data)``: sample lines on the host, parsed, copied
                to the GPU and looked up, as ``examples/test.py`` does

Inputs follow the distributions of ``recflex_amd.workloads`` (bag lengths Poisson, fixed,
truncated normal or lognormal per feature, Zipf or uniform indices, tables N(0, 0.01)), drawn on
the GPU from the seed.
"""

import math

import numpy as np
import torch

from recflex_amd import prebuilt
from recflex_amd.host import RecomHost
from recflex_amd.librecom import RecomLib
from recflex_amd.rec_modules import FeatEmbed, FeatProcessEmbed, RecomModel
from recflex_amd.workloads import Workload, gen_table, row_bytes

MLP_UNITS = [1024, 256, 128]        # examples/end_to_end.py's default
# tables of at most this many rows: C4's full tables (260 GB) fit the card once, not with the
# tables of other seeds beside them
ROW_CAP = 1_000_000


def _case(name, library, batch, entry="bound", bag_scale=1.0, max_rows=ROW_CAP):
    return {"name": name, "library": library, "batch": batch, "entry": entry,
            "bag_scale": bag_scale, "max_rows": max_rows}


def listed():
    return [
        # the smallest model, four features of four lookups: what a call costs
        _case("c1 small call", "c1", 512),
        # a click-through model's categorical features, one lookup each
        _case("c2 one-hot", "c2_tuned", 4096),
        # one request of the 100-feature model with an odd number of candidates, tensors as they come
        _case("c3 request of 37", "c3_tuned", 37, entry="lists"),
        # the 100-feature model at its serving batch: the benchmark's headline workload
        _case("c3 batch", "c3_tuned", 2048),
        # the same model before anyone has tuned it, a ragged batch, from the packed buffer
        _case("c3 untuned, packed", "c3", 1337, entry="packed"),
        # 400 features of fp16 rows, batch scoring: the largest
        _case("c4 fp16 batch", "c4_tuned", 8192),
        # 200 features of int8 rows: quantised inference
        _case("c5 int8 batch", "c5_tuned", 16384),
        # a thousand small features, the reference's own kind of model
        _case("refa thousand features", "refa_tuned", 256),
        # the 100-feature model on traffic with heavy-tailed histories
        _case("c3 skewed lengths", "c3_skew", 2048),
        # few users with very long histories
        _case("few long bags", "fewbags", 16),
        # embedding and MLP end to end
        _case("model c3 with mlp", "c3_tuned", 512, entry="model"),
        # sample lines in, pooled rows out: datasets in the reference's text format
        _case("text lines refa", "refa", 64, entry="text"),
    ]


# what is drawn: library, smallest and largest batch, entries, range of the bag-length factor.  The
# largest cost no more than the listed cases of 8 192 fp16 and 64 lines.
_DRAWN = [
    ("c1", 1, 65536, ("bound", "lists", "packed"), (0.5, 4.0)),
    ("c2_tuned", 1, 65536, ("bound", "lists", "packed"), (1.0, 1.0)),
    ("c3_tuned", 1, 8192, ("bound", "lists", "packed"), (0.25, 2.0)),
    ("c3", 1, 8192, ("bound", "lists", "packed"), (0.25, 2.0)),
    ("c4_tuned", 1, 8192, ("bound", "lists"), (0.25, 1.0)),
    ("c5_tuned", 1, 16384, ("bound", "lists"), (0.25, 1.5)),
    ("refa_tuned", 1, 1024, ("bound", "lists", "packed"), (0.5, 2.0)),
    ("reff4_tuned", 1, 512, ("bound", "packed"), (0.5, 1.0)),
    ("c3_skew", 16, 4096, ("bound", "lists"), (0.5, 1.5)),
    ("fewbags", 1, 256, ("bound", "lists"), (0.02, 1.5)),
    ("c3_tuned", 1, 2048, ("model",), (0.5, 1.5)),
    ("refa_tuned", 1, 512, ("model",), (0.5, 1.5)),
    ("refa", 1, 64, ("text",), (0.5, 1.0)),
]


def draw(rng):
    def log_uniform(lo, hi):
        return math.exp(rng.uniform(math.log(lo), math.log(hi)))

    library, lo, hi, entries, scales = rng.choice(_DRAWN)
    batch = max(lo, min(hi, int(log_uniform(lo, hi + 1))))
    scale = round(log_uniform(*scales), 3)
    if library == "fewbags":                    # as many lookups in all as the listed case, or fewer
        scale = round(min(scale, 24.0 / batch), 3)
    # small tables stay in the caches, large ones do not
    rows = int(log_uniform(20_000, ROW_CAP))
    return {"library": library, "batch": batch, "entry": rng.choice(entries), "bag_scale": scale,
            "max_rows": rows}


# ------------------------------------------------------------------------------------------------

def _workload(case) -> Workload:
    wl = prebuilt.model_spec(case["library"]).workload
    scale = case["bag_scale"]
    feats = []
    for f in wl.features:
        if not prebuilt.is_one_hot(f):
            f = f._replace(mean_bag=f.mean_bag * scale, len_std=f.len_std * scale,
                           len_max=int(math.ceil(f.len_max * scale)))
        feats.append(f._replace(rows=min(f.rows, case["max_rows"])))
    return wl._replace(batch=case["batch"], features=tuple(feats), table_values="normal")


def _bag_lengths(f, batch, g, device):
    """int64 [batch] lengths of one feature's bags."""
    if f.fixed_len:
        lens = torch.full((batch,), int(round(f.mean_bag)), dtype=torch.int64, device=device)
    elif f.len_std > 0:
        # normal truncated at 0 and len_max, by the inverse of its distribution function
        def cdf(x):
            return 0.5 * (1.0 + math.erf((x - f.mean_bag) / (f.len_std * math.sqrt(2.0))))
        lo, hi = cdf(0.0), cdf(f.len_max) if f.len_max > 0 else 1.0
        u = lo + (hi - lo) * torch.rand(batch, generator=g, device=device, dtype=torch.float64)
        z = torch.erfinv((2.0 * u - 1.0).clamp(-1 + 1e-12, 1 - 1e-12))
        lens = (f.mean_bag + f.len_std * math.sqrt(2.0) * z).clamp_(min=0).to(torch.int64)
    elif f.len_sigma > 0:
        mu = math.log(max(f.mean_bag, 0.05)) - f.len_sigma ** 2 / 2
        z = torch.randn(batch, generator=g, device=device, dtype=torch.float64)
        u = torch.rand(batch, generator=g, device=device, dtype=torch.float64)
        lens = torch.floor(torch.exp(mu + f.len_sigma * z) + u).to(torch.int64)
    else:
        mean = torch.full((batch,), float(f.mean_bag), device=device)
        lens = torch.poisson(mean, generator=g).to(torch.int64)
    if f.empty_frac > 0:
        lens[torch.rand(batch, generator=g, device=device) < f.empty_frac] = 0
    return lens


def _indices(f, total, g, device):
    """int32 [total] rows of one feature, Zipf ranks scattered over the table."""
    if f.zipf_alpha <= 0:
        return torch.randint(0, f.rows, (total,), generator=g, device=device, dtype=torch.int32)
    u = torch.rand(total, generator=g, device=device, dtype=torch.float64)
    if abs(f.zipf_alpha - 1.0) < 1e-9:
        rank = float(f.rows) ** u
    else:
        e = 1.0 - f.zipf_alpha
        rank = ((float(f.rows) ** e - 1.0) * u + 1.0) ** (1.0 / e)
    rank = rank.floor_().clamp_(1, f.rows).to(torch.int64)
    a = int(f.rows * 0.6180339887) | 1
    while math.gcd(a, f.rows) != 1:
        a += 2
    return ((rank * a) % f.rows).to(torch.int32)


def _inputs(wl, seed, device):
    g = torch.Generator(device=device)
    g.manual_seed(seed)
    lens = torch.stack([_bag_lengths(f, wl.batch, g, device) for f in wl.features])
    offsets = torch.zeros(len(wl.features), wl.batch + 1, dtype=torch.int32, device=device)
    torch.cumsum(lens, 1, out=lens)
    offsets[:, 1:] = lens
    totals = lens[:, -1].tolist()
    indices = [_indices(f, n, g, device) for f, n in zip(wl.features, totals)]
    return indices, [offsets[k].clone() for k in range(len(wl.features))]


def prepare(case, seed):
    device = torch.device("cuda", torch.cuda.current_device())
    wl = _workload(case)
    entry = case["entry"]
    base = (seed * 1_000_003) % (1 << 31)
    tables = [gen_table(f, base + k, device) for k, f in enumerate(wl.features)]
    indices, offsets = _inputs(wl, base + 500_009, device)
    lib = RecomLib(prebuilt.ensure_built(case["library"]))
    state = {"entry": entry}
    if entry == "text":
        state["layer"] = FeatProcessEmbed(RecomHost(), device, embed_tables=tables, librecom=lib)
        lines = []
        for idx, off in zip(indices, offsets):
            words, cuts = list(map(str, idx.tolist())), off.tolist()
            lines.append([",".join(words[a:b]) for a, b in zip(cuts, cuts[1:])])
        state["lines"] = lines
        return state
    if entry == "model":
        torch.manual_seed(base)
        state["layer"] = RecomModel(MLP_UNITS, device, embed_tables=tables, librecom=lib)
    else:
        state["layer"] = FeatEmbed(device, embed_tables=tables, librecom=lib)
    if entry == "bound":
        state["bound"] = state["layer"].bind_inputs(indices, offsets)
        state["out"] = torch.empty(wl.batch, wl.embed_dim_sum, dtype=torch.float32, device=device)
    elif entry == "lists":
        state["indices"], state["offsets"] = indices, offsets
    else:
        # what FeatPreprocess hands on: (arg_buffers, data_buffer_offsets, scala_args, extra_buffers,
        # extra_buffer_offsets, task_mapping, task_tiles, task_barriers, output_size)
        packed, at = RecomHost().pack([o.cpu().numpy() for o in offsets],
                                      [i.cpu().numpy() for i in indices])
        state["packed"] = (torch.from_numpy(packed).to(device), torch.from_numpy(at).to(device),
                           None, None, None, None, None, None, wl.batch * wl.embed_dim_sum * 4)
    return state


def run(state):
    entry, layer = state["entry"], state["layer"]
    if entry == "bound":
        return layer.forward_indices(state["bound"], out=state["out"])
    if entry == "lists":
        return layer.forward_indices(state["indices"], state["offsets"])
    if entry == "text":
        return layer(state["lines"])
    return layer(*state["packed"])


# ------------------------------------------------------------------------------------------------

def _expected_len(f):
    mean = float(f.mean_bag)
    if f.len_std > 0:
        rng = np.random.default_rng(0)
        z = rng.normal(f.mean_bag, f.len_std, 20_000)
        z = z[(z >= 0) & (z <= (f.len_max or np.inf))]
        mean = float(np.floor(z).mean()) if len(z) else 0.0
    return mean * (1.0 - f.empty_frac)


def _expected_distinct(f, lookups):
    """Rows of the table that ``lookups`` draws touch."""
    if lookups <= 0:
        return 0.0
    if f.zipf_alpha <= 0:
        return f.rows * -math.expm1(-lookups / f.rows)
    # sum over the ranks of 1 - exp(-lookups * p(rank)), on a grid of the rank's logarithm
    edges = np.exp(np.linspace(0.0, math.log(f.rows + 1.0), 1001))
    if abs(f.zipf_alpha - 1.0) < 1e-9:
        cdf = np.log(edges)
    else:
        cdf = (edges ** (1.0 - f.zipf_alpha) - 1.0) / (1.0 - f.zipf_alpha)
    share, ranks = np.diff(cdf) / cdf[-1], np.diff(edges)
    return float(np.sum(ranks * -np.expm1(-lookups * share / ranks)))


def work(case):
    """Every index, offset and touched row read once, every output written once."""
    wl = _workload(case)
    B, nbytes, flops, lookups_in_all, digits = wl.batch, 0.0, 0.0, 0.0, 0.0
    for f in wl.features:
        lookups = B * _expected_len(f)
        nbytes += _expected_distinct(f, lookups) * row_bytes(f.dim, f.data_type)
        nbytes += (B + 1) * 4 + lookups * 4
        flops += lookups * f.dim * (1 if f.data_type != "int8" else 2)
        lookups_in_all += lookups
        digits += lookups * math.log10(max(f.rows, 2))
    if case["entry"] == "text":
        nbytes += digits + lookups_in_all           # the text: digits and separators
    if case["entry"] == "model":
        units = [wl.embed_dim_sum] + MLP_UNITS + [1]
        flops += sum(2.0 * B * a * b for a, b in zip(units, units[1:]))
        nbytes += sum(4.0 * (a * b + b) for a, b in zip(units, units[1:])) + B * 4
    else:
        nbytes += B * wl.embed_dim_sum * 4
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # Against the same sums in 64 bits: fp32 and fp16 rows 0.4e-7 to 1.0e-7, int8 rows 4.3e-7 (a
    # scale and a bias per lookup), the MLP's output 0.4e-7.
    if case["library"] == "c2_tuned":
        return "exact"                              # one lookup per bag: copies of rows
    if case["library"] == "c5_tuned":
        return {"rel": 2e-6}
    return {"rel": 4e-7}
