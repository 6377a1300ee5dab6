"""CPU text front end (librecflex_host.so, recom_host_* in include/recflex_hip.h) against the
oracle's restatement of the reference's line splitter, plus the packed-buffer layout."""

import os
import shutil
import sys

import numpy as np
import pytest

from helpers import oracle
from recflex_amd.code_emitter import CodeEmitter, MetaData
from recflex_amd.code_emitter.build_basic import BasicBuilder
from recflex_amd.host import RecomHost, RecomHostError
from recflex_amd.model_build import default_feat_schedules
from recflex_amd.utils import compile_build


@pytest.fixture(scope="module")
def host():
    return RecomHost(BasicBuilder().build())


CASES = [
    ["3,5,7", "", "12", "0", "1,,2", "9,", ",4", "007", "1 2;3"],
    [""],
    ["", "", ""],
    ["5"],
    ["1,2", ""],
    ["", "1,2"],
    [],
    ["2147483647", "0"],
]


@pytest.mark.parametrize("lines", CASES)
def test_parse_matches_oracle(host, lines):
    idx, off = host.parse_lines(lines)
    want_idx, want_off = oracle.parse_lines_python(lines)
    assert idx.dtype == np.int32 and off.dtype == np.int32
    assert np.array_equal(idx, want_idx)
    assert np.array_equal(off, want_off)


def test_parse_random_against_both_oracles(host):
    rng = np.random.default_rng(10)
    seps = [",", " ", ";", ",,"]
    lines = []
    for _ in range(500):
        n = int(rng.integers(0, 15))
        sep = seps[int(rng.integers(0, len(seps)))]
        lines.append(sep.join(str(int(v)) for v in rng.integers(0, 2 ** 31 - 1, n)))
    idx, off = host.parse_lines(lines)
    for want_idx, want_off in (oracle.parse_lines_python(lines), oracle.parse_lines_c(lines)):
        assert np.array_equal(idx, want_idx) and np.array_equal(off, want_off)


def test_parse_rejects_values_beyond_int32(host):
    with pytest.raises(RecomHostError):
        host.parse_lines(["2147483648"])


def test_raw_entry_point_error_codes(host):
    import ctypes
    lib = host.lib
    off = (ctypes.c_int32 * 3)()
    idx = (ctypes.c_int32 * 8)()
    n = ctypes.c_int64()
    # capacity too small
    assert lib.recom_host_parse_lines(b"1,2", 3, 1, idx, 1, off, ctypes.byref(n)) == -2
    # more lines than announced / fewer lines than announced
    assert lib.recom_host_parse_lines(b"1\n2\n3", 5, 2, idx, 8, off, ctypes.byref(n)) == -3
    assert lib.recom_host_parse_lines(b"1", 1, 2, idx, 8, off, ctypes.byref(n)) == -3
    # NULL outputs
    assert lib.recom_host_parse_lines(b"1", 1, 1, idx, 1, None, ctypes.byref(n)) == -1
    # one trailing newline after the last line is fine
    assert lib.recom_host_parse_lines(b"7\n", 2, 1, idx, 1, off, ctypes.byref(n)) == 0
    assert (n.value, idx[0], off[0], off[1]) == (1, 7, 0, 1)


def test_alignment_helpers(host):
    """128-byte alignment of utils.cuh:60-68."""
    assert [host.alignmem(x) for x in (0, 1, 127, 128, 129, 4 * 513)] == [0, 128, 128, 128, 256, 2176]


def test_pack_layout(host):
    rng = np.random.default_rng(11)
    batch = 37
    offsets, indices = [], []
    for f in range(5):
        lens = rng.integers(0, 6, batch)
        if f == 3:
            lens[:] = 0          # a feature without any lookup
        off = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
        offsets.append(off)
        indices.append(rng.integers(0, 1000, off[-1]).astype(np.int32))
    packed, byte_offsets = host.pack(offsets, indices)
    assert packed.dtype == np.int32 and byte_offsets.dtype == np.int64
    assert byte_offsets[0] == 0 and len(byte_offsets) == 6
    raw = packed.view(np.uint8)
    for f in range(5):
        start = int(byte_offsets[f])
        assert start % 128 == 0
        off_bytes = (batch + 1) * 4
        got_off = raw[start:start + off_bytes].view(np.int32)
        assert np.array_equal(got_off, offsets[f])
        idx_start = start + host.alignmem(off_bytes)
        got_idx = raw[idx_start:idx_start + 4 * len(indices[f])].view(np.int32)
        assert np.array_equal(got_idx, indices[f])
        # padding is zero
        assert not raw[start + off_bytes:idx_start].any()
        end = int(byte_offsets[f + 1])
        assert end == idx_start + host.alignmem(4 * len(indices[f]))
        assert not raw[idx_start + 4 * len(indices[f]):end].any()
    assert int(byte_offsets[-1]) == raw.size


def test_preprocess_tuple_shape(host):
    raw = [["1,2", "", "3"], ["4", "5", "6"]]
    (dbo, out_off, extra_off, task_mapping, task_tiles, data, scala) = host.preprocess(raw, 0)
    assert len(dbo) == 3 and dbo[0] == 0
    assert extra_off == [0, 0, 0] and task_mapping == [] and task_tiles == [0, 0]
    assert scala == [3, 3, 3, 3]                      # (num_inputs, num_segments) per feature
    assert data[0].tolist() == [0, 2, 2, 3] and data[1].tolist() == [1, 2, 3]
    assert data[2].tolist() == [0, 1, 2, 3] and data[3].tolist() == [4, 5, 6]


def _feature_lines(rng, batch, mean):
    return [",".join(str(int(v)) for v in rng.integers(0, 2 ** 31 - 1, rng.poisson(mean))) for _ in range(batch)]


@pytest.mark.parametrize("features, batch, mean", [(1, 0, 0.), (1, 1, 3.), (5, 33, 0.3), (3, 31, 12.),
                                                   (40, 64, 60.), (2, 1500, 40.)])
def test_joint_parse_equals_feature_by_feature(host, features, batch, mean):
    """One thread and several (128 KiB of text each), offsets that end on a 128-byte boundary and not,
    separators of other kinds, empty lines."""
    rng = np.random.default_rng(features * 1000 + batch)
    raw = [_feature_lines(rng, batch, mean) for _ in range(features)]
    if batch > 8:
        raw[0][:8] = ["", "1,,2", "9,", ",4", ";", "é5", "", "007"]
    dbo, _, _, _, _, data, scala = host.preprocess(raw)
    packed = host.packed.copy()
    want_data, want_scala, want_offsets = host._parse_each(raw)
    assert np.array_equal(packed, host.packed) and dbo == want_offsets.tolist() and scala == want_scala
    assert len(data) == len(want_data) and all(
        a.dtype == np.int32 and np.array_equal(a, b) for a, b in zip(data, want_data))


@pytest.mark.parametrize("features, batch", [(3, 31), (1, 1), (12, 64)])
def test_preprocess_data_are_arrays_of_their_own(host, features, batch):
    """Changing ``data`` changes neither the packed buffer nor one another, and none of them, nor
    the packed buffer, holds on to more memory than its own."""
    rng = np.random.default_rng(5)
    raw = [_feature_lines(rng, batch, 9.) for _ in range(features)]
    data = host.preprocess(raw)[5]
    packed, before = host.packed, host.packed.copy()
    assert packed.base is None and packed.flags.owndata
    for k, a in enumerate(data):
        assert a.base is None and a.flags.owndata and a.flags.writeable
        a[:] = -1 - k
    assert np.array_equal(packed, before)
    assert all((a == -1 - k).all() for k, a in enumerate(data))


def test_feat_preprocess_takes_any_host(host):
    """The host as it is, a subclass and an instance with a ``preprocess`` of their own: the same
    tensors, and the caller's ``preprocess`` runs."""
    import torch
    from recflex_amd.host import RecomHost
    from recflex_amd.rec_modules import FeatPreprocess

    class Own(RecomHost):
        def preprocess(self, raw_data, max_concurrent_blocks=0):
            calls.append(max_concurrent_blocks)
            return super().preprocess(raw_data, max_concurrent_blocks)

    calls = []
    rng = np.random.default_rng(6)
    raw = [_feature_lines(rng, 21, 7.) for _ in range(4)]
    own, patched = Own(), RecomHost()
    patched.preprocess = own.preprocess
    patched.packed = None
    want = FeatPreprocess(RecomHost(), torch.device("cpu"), output_units=8)(raw, 5)
    got = FeatPreprocess(own, torch.device("cpu"), output_units=8)(raw, 5)
    data = FeatPreprocess(patched, torch.device("cpu"), output_units=8)(raw, 6)[0]
    assert calls == [5, 6] and len(want) == len(got) == 9 and want[-1] == got[-1] == 21 * 8 * 4
    assert all(torch.equal(a, b) for a, b in zip(want[:-1], got[:-1]))
    # no packed buffer: the arrays of data, one after the other
    assert data.tolist() == np.concatenate(own.preprocess(raw)[5]).tolist()


@pytest.mark.parametrize("bad, message", [({2: "2147483648", 4: "1\n2"}, "int32"), ({3: "1\n2\n3", 4: "99999999999"}, "lines")])
def test_joint_parse_reports_the_first_feature_that_fails(host, bad, message):
    raw = [["1,2", "3"] for _ in range(6)]
    for f, text in bad.items():
        raw[f][0] = text
    for parse in (host.preprocess, host._parse_each):
        with pytest.raises(RecomHostError, match=message):
            parse(raw)


# lists, tuples and what only the joined text can hold; lengths around the eight bytes that are read at a time,
# numbers of up to ten digits, separators at the ends
@pytest.mark.parametrize("line", ["", "5", ",", "1234567", "12345678", "1234567,", ",1234567", "123456,89012345", "2147483647",
                                  "0,00000000007,1", "9;8 7\t6", "12345678,87654321,1", "1,2,3,4,5,6,7,8", "é,1", "1,₂,3"])
@pytest.mark.parametrize("box", [list, tuple])
def test_strings_where_they_lie_equal_the_joined_text(host, line, box):
    if host._strings is None:
        pytest.skip("the library was built without the reader of strings, or for another interpreter")
    raw = box([box([line, "1", line, "", line + line]), box(["7", "", "8,9", line, ""])])
    if max((len(w) for w in line.replace(";", ",").split(",")), default=0) > 5:
        raw = box([box([line, "1", line, "", line]), box(["7", "", "8,9", line, ""])])
    counts, at = np.empty(2, np.int64), np.zeros(3, np.int64)
    want = host._parse_joined(raw, 5, counts, at)
    got_counts, got_at = np.empty(2, np.int64), np.zeros(3, np.int64)
    got = host._parse_strings(raw, 5, got_counts, got_at)
    if not line.isascii():
        assert got is None
    else:
        assert np.array_equal(got, want) and np.array_equal(got_counts, counts) and np.array_equal(got_at, at)
    assert np.array_equal(host._parse_packed(list(raw), False)[2], at) and np.array_equal(host.packed, want)


def test_strings_that_are_not_plain_are_left_to_the_joined_text(host):
    class Line(str):
        pass

    counts, at = np.empty(1, np.int64), np.zeros(2, np.int64)
    for lines in (["1\n2", "3"], ["2147483648", "1"], ["99999999999", "1"], [Line("1"), "2"], [b"1", "2"], np.array(["1", "2"]),
                  ["1"], [None, "1"]):
        assert host._parse_strings([lines], 2, counts, at) is None
    assert host._parse_strings(np.array([["1", "2"]]), 2, counts, at) is None


def test_a_generated_library_reads_the_strings_where_they_lie(tmp_path, host):
    """``recom_host.so`` as a model's CMake project builds it, the library that the examples load."""
    if host._strings is None:
        pytest.skip("no reader of strings for this interpreter")
    fs = default_feat_schedules([MetaData(8, "float"), MetaData(16, "half")], [3.0, 5.0])
    emitter = CodeEmitter(fs)
    emitter.emit_host(str(tmp_path / "preprocess.cpp"))
    emitter.emit_cmake_list(str(tmp_path / "CMakeLists.txt"), code_fname=None, host_fname="preprocess.cpp")
    compile_build(str(tmp_path / "build"))
    generated = RecomHost(str(tmp_path / "build" / "recom_host.so"))
    raw = [["1,2", "", "3"], ["4", "5,6,7", ""]]
    counts, at = np.empty(2, np.int64), np.zeros(3, np.int64)
    got = generated._parse_strings(raw, 3, counts, at)
    assert got is not None and np.array_equal(got, host._parse_joined(raw, 3, counts.copy(), at.copy()))


@pytest.fixture
def builder(tmp_path):
    b = BasicBuilder()
    (tmp_path / "host").mkdir()
    for name in ("host_source", "strings_source"):
        setattr(b, name, shutil.copy(getattr(b, name), tmp_path / "host"))
    b.csrc_dir = str(tmp_path)
    return b


def test_host_library_follows_its_sources(builder, monkeypatch):
    """Built when it is missing, kept as long as sources, flags and interpreter are what it was built from."""
    def edit(path):
        with open(path, "a") as f:
            f.write("\n// edited\n")

    lib = builder.build()
    steps = [(lambda: None, False), (lambda: edit(builder.host_source), True), (lambda: None, False),
             (lambda: builder.host_flags.append("-DX"), True)]
    if builder.strings_build():
        steps += [(lambda: edit(builder.strings_source), True),
                  (lambda: monkeypatch.setattr(sys.implementation, "cache_tag", "cpython-000"), True)]
    for change, again in steps + [(lambda: None, False)]:
        change()
        built = os.stat(lib).st_ino
        assert builder.build() == lib and (os.stat(lib).st_ino != built) is again
    os.unlink(lib + ".from")                        # a library of before this was kept
    built = os.stat(lib).st_ino
    builder.build()
    assert os.stat(lib).st_ino != built
    builder.cxx = "/no/such/compiler"
    builder.build()
    builder.host_flags.append("-DY")
    with pytest.warns(RuntimeWarning, match="could not be built again"):
        assert builder.build() == lib


def test_a_string_reader_that_does_not_compile_is_named(builder):
    if not builder.strings_build():
        pytest.skip("no Python headers")
    with open(builder.strings_source, "a") as f:
        f.write("not c++\n")
    with pytest.warns(RuntimeWarning, match="not c"):
        host = RecomHost(builder.build())
    assert host._strings is None and np.array_equal(host.parse_lines(["1,2"])[0], [1, 2])


def test_another_interpreters_strings_are_not_read(host, monkeypatch):
    """Of another version, or with other objects (sys.getobjects is there if they begin with links)."""
    if host._strings is None:
        pytest.skip("no reader of strings for this interpreter")
    assert RecomHost(host.path)._strings is not None
    with monkeypatch.context() as m:
        m.setattr(sys, "getobjects", lambda n: [], raising=False)
        assert RecomHost(host.path)._strings is None
    monkeypatch.setattr(sys, "version_info", (3, 99, 0))
    assert RecomHost(host.path)._strings is None
