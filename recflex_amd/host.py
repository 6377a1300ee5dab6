"""ctypes bindings of the CPU text front end (``recom_host_*`` in ``include/recflex_hip.h``).

``RecomHost`` stands where the reference has the generated pybind module ``recom_host``
(``RecFlex/code_emitter/codegen.py:90-218``): ``preprocess(raw_data, max_concurrent_blocks)``
takes the ``List[F][B]`` of sample lines and returns a 7-tuple in the reference's order
``(data_buffer_offsets, output_offsets, extra_buffer_offsets, task_mapping, task_tiles, data,
scala_data)``.  Differences, all consequences of the device-side thread binding:
``task_mapping`` is empty and ``task_tiles`` is zero (tiles are decided on the GPU),
``extra_buffer_offsets`` is all zero (no schedule needs scratch memory), ``data`` holds numpy
int32 arrays ``[offsets_0, indices_0, offsets_1, indices_1, ...]`` instead of Python lists, and
inside the packed buffer a feature's offsets come first, then its indices.
"""

import ctypes
import os
import sys
from typing import List, Sequence, Tuple

import numpy as np

_I32P = ctypes.POINTER(ctypes.c_int32)
_I64P = ctypes.POINTER(ctypes.c_int64)

_ERRORS = {-1: "invalid argument", -2: "output capacity too small",
           -3: "text holds a different number of lines than expected",
           -4: "index does not fit in int32"}


class RecomHostError(RuntimeError):
    pass


def _declare(lib: ctypes.CDLL) -> None:
    lib.recom_host_parse_lines.restype = ctypes.c_int
    lib.recom_host_parse_lines.argtypes = [ctypes.c_char_p, ctypes.c_int64, ctypes.c_int32, _I32P,
                                           ctypes.c_int64, _I32P, _I64P]
    lib.recom_host_max_indices.restype = ctypes.c_int64
    lib.recom_host_max_indices.argtypes = [ctypes.c_int64]
    lib.recom_host_alignmem.restype = ctypes.c_int64
    lib.recom_host_alignmem.argtypes = [ctypes.c_int64]
    lib.recom_host_packed_size.restype = ctypes.c_int64
    lib.recom_host_packed_size.argtypes = [ctypes.c_int32, ctypes.c_int64]
    lib.recom_host_pack.restype = ctypes.c_int
    lib.recom_host_pack.argtypes = [ctypes.c_int32, ctypes.c_int32, ctypes.POINTER(_I32P),
                                    ctypes.POINTER(_I32P), _I64P, ctypes.c_void_p, ctypes.c_int64, _I64P]
    if hasattr(lib, "recom_host_parse_packed"):
        lib.recom_host_parse_packed.restype = ctypes.c_int
        lib.recom_host_parse_packed.argtypes = [ctypes.c_int32, ctypes.c_int32,
                                                ctypes.POINTER(ctypes.c_char_p), _I64P, ctypes.c_void_p,
                                                ctypes.c_int64, _I64P, _I64P]


def _string_reader(path: str):
    """The library once more, for calls that keep the interpreter's lock, if it reads the strings of
    this interpreter (``csrc/host/recflex_strings.cpp``); ``None`` otherwise."""
    lib = ctypes.PyDLL(path)
    if sys.implementation.name != "cpython" or not hasattr(lib, "recom_host_parse_strings") \
            or getattr(sys, "_is_gil_enabled", lambda: True)() is False \
            or lib.recom_host_strings_python() != sys.version_info[0] * 256 + sys.version_info[1] \
            + (65536 if hasattr(sys, "getobjects") else 0):
        return None
    lib.recom_host_count_strings.restype = ctypes.c_int
    lib.recom_host_count_strings.argtypes = [ctypes.py_object, ctypes.c_int32, ctypes.c_int32, ctypes.c_void_p]
    lib.recom_host_parse_strings.restype = ctypes.c_int
    lib.recom_host_parse_strings.argtypes = [ctypes.py_object, ctypes.c_int32, ctypes.c_int32, ctypes.c_void_p,
                                             ctypes.c_void_p, ctypes.c_int64, ctypes.c_void_p]
    return lib


def default_host_lib_path() -> str:
    from recflex_amd.code_emitter.build_basic import BasicBuilder
    return BasicBuilder().host_lib_path()


class RecomHost:
    """Loads ``librecflex_host.so`` (model independent) or a generated ``recom_host.so``
    (which also knows the model's feature count)."""

    def __init__(self, path: str = None):
        self.path = path or default_host_lib_path()
        if not os.path.exists(self.path):
            raise FileNotFoundError(
                f"{self.path} is not built; run recflex_amd.code_emitter.build_basic.BasicBuilder().build()")
        self.lib = ctypes.CDLL(self.path)
        _declare(self.lib)
        self.num_features = None
        if hasattr(self.lib, "recom_host_num_features"):
            self.lib.recom_host_num_features.restype = ctypes.c_int32
            self.num_features = int(self.lib.recom_host_num_features())
        self._strings = _string_reader(self.path)
        self._knows_dims = hasattr(self.lib, "recom_host_output_row_bytes")
        if self._knows_dims:
            self.lib.recom_host_output_row_bytes.restype = ctypes.c_int64
            self.lib.recom_host_output_row_bytes.argtypes = [ctypes.c_int32]

    # -------------------------------------------------------------------------------------

    def parse_lines(self, lines: Sequence[str]) -> Tuple[np.ndarray, np.ndarray]:
        """Sample lines of one feature -> (indices int32[L], offsets int32[B+1])."""
        text = "\n".join(lines).encode()
        n_lines = len(lines)
        cap = int(self.lib.recom_host_max_indices(len(text)))
        indices = np.empty(max(cap, 1), dtype=np.int32)
        offsets = np.empty(n_lines + 1, dtype=np.int32)
        n = ctypes.c_int64(0)
        rc = self.lib.recom_host_parse_lines(text, len(text), n_lines,
                                             indices.ctypes.data_as(_I32P), cap,
                                             offsets.ctypes.data_as(_I32P), ctypes.byref(n))
        if rc != 0:
            raise RecomHostError(f"recom_host_parse_lines: {_ERRORS.get(rc, rc)}")
        return indices[:n.value].copy(), offsets

    def alignmem(self, nbytes: int) -> int:
        return int(self.lib.recom_host_alignmem(nbytes))

    def pack(self, offsets: List[np.ndarray], indices: List[np.ndarray]) -> Tuple[np.ndarray, np.ndarray]:
        """Per-feature arrays -> (packed int32 buffer, int64 byte offsets [F+1])."""
        num_feats = len(offsets)
        assert len(indices) == num_feats
        if num_feats == 0:
            return np.zeros(0, dtype=np.int32), np.zeros(1, dtype=np.int64)
        batch = len(offsets[0]) - 1
        offs = [np.ascontiguousarray(o, dtype=np.int32) for o in offsets]
        idxs = [np.ascontiguousarray(i, dtype=np.int32) for i in indices]
        for o in offs:
            if len(o) != batch + 1:
                raise ValueError("all features must have the same batch size")
        counts = np.array([len(i) for i in idxs], dtype=np.int64)
        total = sum(int(self.lib.recom_host_packed_size(batch, int(c))) for c in counts)
        dst = np.empty(total // 4, dtype=np.int32)
        byte_offsets = np.zeros(num_feats + 1, dtype=np.int64)
        off_ptrs = (_I32P * num_feats)(*[o.ctypes.data_as(_I32P) for o in offs])
        idx_ptrs = (_I32P * num_feats)(*[i.ctypes.data_as(_I32P) for i in idxs])
        rc = self.lib.recom_host_pack(num_feats, batch, off_ptrs, idx_ptrs,
                                      counts.ctypes.data_as(_I64P), dst.ctypes.data_as(ctypes.c_void_p),
                                      total, byte_offsets.ctypes.data_as(_I64P))
        if rc != 0:
            raise RecomHostError(f"recom_host_pack: {_ERRORS.get(rc, rc)}")
        return dst, byte_offsets

    # -------------------------------------------------------------------------------------

    def _parse_packed(self, raw_data: List[List[str]], with_data: bool
                      ) -> Tuple[List[np.ndarray], np.ndarray, np.ndarray]:
        """Sets ``self.packed``; returns ``data`` (empty unless asked for), ``scala_data`` and the
        packed buffer's byte offsets.  Native calls for all features on several threads, each
        feature parsed straight into its place: a thousand features of 64 lines, 3.7 MB of text,
        take 0.9 ms read from the strings where they lie and 2.3 ms by way of a joined and encoded
        text per feature."""
        num_feats = len(raw_data)
        batches = {len(lines) for lines in raw_data}
        if len(batches) != 1 or not hasattr(self.lib, "recom_host_parse_packed"):
            data, scala, byte_offsets = self._parse_each(raw_data)
            return data, np.array(scala, dtype=np.int32), byte_offsets
        batch = batches.pop()
        off_bytes = self.alignmem((batch + 1) * 4)
        byte_offsets = np.zeros(num_feats + 1, dtype=np.int64)
        counts = np.empty(num_feats, dtype=np.int64)
        dst = self._parse_strings(raw_data, batch, counts, byte_offsets)
        if dst is None:
            dst = self._parse_joined(raw_data, batch, counts, byte_offsets)
        self.packed = dst
        scala_data = np.stack([counts, np.full(num_feats, batch)], 1).ravel().astype(np.int32)  # num_inputs, num_segments
        data: List[np.ndarray] = []
        if with_data:
            # arrays of their own: a caller may change them without changing what goes to the GPU,
            # and one that is kept keeps nothing else alive
            for at, n in zip((byte_offsets[:-1] // 4).tolist(), counts.tolist()):
                first = at + off_bytes // 4
                data += [dst[at:at + batch + 1].copy(), dst[first:first + n].copy()]
        return data, scala_data, byte_offsets

    def _parse_strings(self, raw_data, batch: int, counts: np.ndarray, byte_offsets: np.ndarray):
        """The packed buffer, read from the strings where they lie; ``None``: they are not plain ASCII
        strings in lists, or hold what only the other path knows what to say to."""
        if self._strings is None:
            return None
        num_feats = len(raw_data)
        if self._strings.recom_host_count_strings(raw_data, num_feats, batch, counts.ctypes.data) != 0:
            return None
        size = num_feats * self.alignmem((batch + 1) * 4) + int((((counts * 4) + 127) // 128 * 128).sum())
        dst = np.empty(size // 4, dtype=np.int32)
        if self._strings.recom_host_parse_strings(raw_data, num_feats, batch, counts.ctypes.data, dst.ctypes.data,
                                                  dst.nbytes, byte_offsets.ctypes.data) != 0:
            return None
        return dst

    def _parse_joined(self, raw_data, batch: int, counts: np.ndarray, byte_offsets: np.ndarray) -> np.ndarray:
        """The packed buffer by way of one text per feature."""
        num_feats = len(raw_data)
        texts = ["\n".join(lines).encode() for lines in raw_data]
        lens = np.array([len(t) for t in texts], dtype=np.int64)
        # room for the most indices such texts can hold; pages that stay empty are never touched
        capacity = int(num_feats * (self.alignmem((batch + 1) * 4) + 128) + 4 * (lens + 1).sum())
        dst = np.empty((capacity + 3) // 4, dtype=np.int32)
        rc = self.lib.recom_host_parse_packed(num_feats, batch, (ctypes.c_char_p * num_feats)(*texts),
                                              lens.ctypes.data_as(_I64P), dst.ctypes.data_as(ctypes.c_void_p),
                                              dst.nbytes, byte_offsets.ctypes.data_as(_I64P),
                                              counts.ctypes.data_as(_I64P))
        if rc != 0:
            raise RecomHostError(f"recom_host_parse_lines: {_ERRORS.get(rc, rc)}")
        dst.resize(int(byte_offsets[-1]) // 4, refcheck=False)      # gives the rest of the room back
        return dst

    def _parse_each(self, raw_data: List[List[str]]) -> Tuple[List[np.ndarray], List[int], np.ndarray]:
        """The same, feature by feature: no features, lists of unequal length (an error unless a
        line fails to parse first), or a generated library from before the joint call."""
        offsets, indices = [], []
        data: List[np.ndarray] = []
        scala_data: List[int] = []
        for lines in raw_data:
            idx, off = self.parse_lines(lines)
            offsets.append(off)
            indices.append(idx)
            data.extend([off, idx])
            scala_data.extend([len(idx), len(off) - 1])   # num_inputs, num_segments
        self.packed, byte_offsets = self.pack(offsets, indices)
        return data, scala_data, byte_offsets

    def _check_features(self, raw_data) -> None:
        if self.num_features is not None and len(raw_data) != self.num_features:
            raise ValueError(f"this host library was generated for {self.num_features} features, "
                             f"got {len(raw_data)}")

    def _output_row_bytes(self, feature: int) -> int:
        return int(self.lib.recom_host_output_row_bytes(feature)) if self._knows_dims else 0

    def preprocess(self, raw_data: List[List[str]], max_concurrent_blocks: int = 0):
        num_feats = len(raw_data)
        self._check_features(raw_data)
        data, scala_data, byte_offsets = self._parse_packed(raw_data, True)
        data_buffer_offsets = byte_offsets.tolist()
        # byte offsets of each feature's slab of pooled output (prefix sum of batch * dim * 4,
        # reference: codegen.py:144-147); the generic library does not know the dims and
        # reports zeros, FeatPreprocess then sizes the output from the model's dims
        output_offsets = [0]
        for f, lines in enumerate(raw_data):
            output_offsets.append(output_offsets[-1] + len(lines) * self._output_row_bytes(f))
        extra_buffer_offsets = [0] * (num_feats + 1)
        task_mapping: List[Tuple[int, int]] = []
        task_tiles = [0] * num_feats
        return (data_buffer_offsets, output_offsets, extra_buffer_offsets, task_mapping,
                task_tiles, data, scala_data.tolist())

    def preprocess_packed(self, raw_data: List[List[str]]) -> Tuple[np.ndarray, int, np.ndarray]:
        """What ``FeatPreprocess`` needs of ``preprocess``, as arrays: sets ``self.packed``, returns
        the byte offsets of the features (int64 [F+1]), the bytes of pooled output if the library
        knows the dims (else 0), and num_inputs, num_segments per feature (int32 [2F])."""
        self._check_features(raw_data)
        _, scala_data, byte_offsets = self._parse_packed(raw_data, False)
        output_size = sum(len(lines) * self._output_row_bytes(f) for f, lines in enumerate(raw_data)) \
            if self._knows_dims else 0
        return byte_offsets, output_size, scala_data
