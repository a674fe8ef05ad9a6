"""CPU-only checks of the boundary: the shared library loads and exports every
entry point declared in include/trigrad_hip.h, rejects bad arguments before
touching a device, and the Python layer raises the reference's exceptions."""
import ctypes as C
import os
import re

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _declared_entry_points():
    text = open(os.path.join(ROOT, "include", "trigrad_hip.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(tg_[a-z0-9_]+)\s*\(", text)))


@pytest.mark.parametrize("bits", [32, 64])
def test_library_exports_every_declared_entry_point(bits):
    """Both builds of the library (float, and double = the reference's DOUBLE_PRECISION)."""
    from trigrad_amd import _lib
    lib = _lib.load(bits)
    names = _declared_entry_points()
    assert len(names) >= 14
    for name in names:
        assert hasattr(lib, name), f"{name} is declared in include/trigrad_hip.h but not exported"
    assert sorted(_lib.SIGNATURES) == names, "trigrad_amd/_lib.py must declare exactly the header's entry points"
    assert lib.tg_version() == 1
    assert lib.tg_precision_bits() == bits


@pytest.mark.parametrize("tile_w,tile_h,at_once_32,at_once_23", [
    (8, 8, 9, 11), (2, 2, 9, 11), (8, 16, 5, 7), (12, 16, 3, 5), (16, 16, 3, 4), (20, 13, 3, 4),
])
def test_candidate_places_save_a_generation_of_workgroups(tile_w, tile_h, at_once_32, at_once_23):
    """at_once: workgroups a CU with 32 and with 23 places of 6 bytes a thread in LDS next to 64 staged records of 64 bytes: by
    160 KB of LDS in pieces of 1280 bytes, and by three and four waves a SIMD, which the kernels are compiled for."""
    from trigrad_amd import _lib
    lib = _lib.load(32)
    threads = -(-tile_w * tile_h // 64) * 64
    split = -(-tile_w * tile_h // min(threads, 256))  # workgroups of a tile
    threads = min(threads, 256)
    for places, at_once, waves in ((32, at_once_32, 3), (23, at_once_23, 4)):
        pieces = -(-(64 * 64 + places * threads * 6 + 512) // 1280)
        assert at_once == min(128 // pieces, waves * 256 // threads)
    for tiles in sorted({256 * n * k + d for n in (at_once_32, at_once_23) for k in (1, 2, 3) for d in (-1, 0, 1)}):
        groups = split * tiles
        generations = [-(-groups // (256 * n)) for n in (at_once_32, at_once_23)]
        assert lib.tg_candidate_places(tile_w * tiles, tile_h, tile_w, tile_h) == (32 if generations[0] <= generations[1] else 23)
    assert lib.tg_candidate_places(0, 16, 16, 16) == 0 and lib.tg_candidate_places(64, 64, 64, 32) == 0
    assert _lib.load(64).tg_candidate_places(8192, 8192, 16, 16) == 32


@pytest.mark.parametrize("bits", [32, 64])
def test_host_side_helpers_and_argument_rejection(bits):
    from trigrad_amd import _lib
    lib = _lib.load(bits)
    assert lib.tg_num_tiles(1920, 1080, 16, 16) == 120 * 68
    assert lib.tg_num_tiles(50, 50, 4, 4) == 13 * 13
    assert lib.tg_num_tiles(0, 10, 16, 16) == 0
    assert lib.tg_scan_workspace_bytes(0) > 0 and lib.tg_scan_workspace_bytes(10 ** 6) < 10 ** 5
    assert lib.tg_sort_workspace_bytes(1 << 30) == 0  # more pairs than the 30-bit look-back counters hold
    assert lib.tg_sort_workspace_bytes(10 ** 6) > 0
    # rejected before any device work: negative sizes, null pointers, oversized tiles
    assert lib.tg_bin_count(None, 0, None, -1, 64, 64, 16, 16, None, None) == -1
    assert b"tg_bin_count" in lib.tg_last_error()
    assert lib.tg_bin_count(None, 3, None, 5, 64, 64, 16, 16, None, None) == -1
    assert lib.tg_bin_count(None, 0, None, 0, 64, 64, 16, 16, None, None) == 0  # nothing to do
    assert lib.tg_scan_exclusive_u32(None, None, 8, None, None, 0, None, 256, 0, None, None) == -1
    res = C.c_int(7)
    assert lib.tg_sort_pairs_u64_u32(None, None, None, None, 1 << 31, 64, None, 0, None, C.byref(res), None) == -1
    assert lib.tg_tile_ranges(None, 5, 10, None, None) == -1
    assert lib.tg_render_forward(*([None] * 7), 64, 64, 64, 32, 0.0, 0, 1, *([None] * 12)) == -1
    assert b"tile_w*tile_h" in lib.tg_last_error()
    assert lib.tg_render_forward(*([None] * 7), 64, 64, 16, 16, 0.0, 0, 0, *([None] * 12)) == -1
    assert b"max_layers" in lib.tg_last_error()
    assert lib.tg_render_backward(*([None] * 17), 64, 64, 16, 16, 0.0, 0, 1, None, None, None, 4, 3, 1, None) == -1
    assert lib.tg_split_gradient_block(None, 5, None, None, None, None) == -1 and b"null pointer" in lib.tg_last_error()
    assert lib.tg_split_gradient_block(None, -1, None, None, None, None) == -1
    assert lib.tg_split_gradient_block(None, 0, None, None, None, None) == 0
    assert lib.tg_hit_mask_words(6400, 64, 64, 16, 16) == 16 + (100 + 16 + 1) * 256  # a word per workgroup, then the chunks
    assert lib.tg_list_bound_words(6400, 16) == 25 + 16 + 1
    assert lib.tg_list_bounds(None, 0, None, 0, None, None, None, 0, None, None, None, None) == -1
    # the frame's two calls and the tile-list sort
    assert lib.tg_bin_setup_workspace_bytes(10 ** 6, 1920, 1080, 16, 16) % 256 == 0
    assert 0 < lib.tg_bin_setup_workspace_bytes(0, 64, 64, 16, 16) < 10 ** 4
    assert lib.tg_bin_setup_workspace_bytes(-1, 64, 64, 16, 16) == 0
    assert lib.tg_bin_setup(None, 0, None, 5, 64, 64, 16, 16, None, None, None, 0, None, None, 0, None) == -1
    assert b"tg_bin_setup" in lib.tg_last_error()
    assert lib.tg_build_tile_lists_workspace_bytes(10 ** 6, 8160) > 0 and lib.tg_build_tile_lists_workspace_bytes(1 << 30, 8160) == 0
    assert lib.tg_tile_list_sort_workspace_bytes(10 ** 6, 0) == 0
    res = C.c_int(7)
    assert lib.tg_build_tile_lists(None, None, 5, 10, 0, None, None, 64, 64, 16, 16, None, None, None, None, None, None, 0, None, 0,
                                   C.byref(res), None) == -1
    assert lib.tg_sort_tile_lists(None, None, None, None, 10, 0, None, None, 0, None, C.byref(res), None) == -1
    # the frame's binning without a wait for the host (float build) and the sort of its keys
    assert lib.tg_bin_frame_supported(1920, 1080, 16, 16) == (1 if bits == 32 else 0)
    assert lib.tg_bin_frame_supported(1 << 14, 1 << 14, 2, 2) == 0  # more than 2^21 tiles
    assert lib.tg_bin_frame_workspace_bytes(10 ** 6, 3 * 10 ** 6, 1920, 1080, 16, 16) % 256 == 0
    assert lib.tg_bin_frame_workspace_bytes(10 ** 6, 3 * 10 ** 6, 1920, 1080, 16, 16) > 52 * 10 ** 6  # records and offsets of the triangles
    assert lib.tg_bin_frame_workspace_bytes(-1, 0, 64, 64, 16, 16) == 0
    assert lib.tg_bin_frame(None, 0, None, 5, 64, 64, 16, 16, None, None, 0, None, None, 0, 1, None, 0, None, None) == -1
    assert b"tg_bin_frame" in lib.tg_last_error()
    assert lib.tg_build_frame_lists_workspace_bytes(10 ** 6, 120, 68) > 0 and lib.tg_build_frame_lists_workspace_bytes(1 << 30, 120, 68) == 0
    assert lib.tg_build_frame_lists(None, 1, 10, 120, 68, None, None, None, None, None, None, 0, None, C.byref(res), None) == -1
    lib.tg_force_tickets(1)
    lib.tg_force_tickets(0)
    assert lib.tg_scan_noalloc_max_n() == 1 << 24
    assert lib.tg_scan_exclusive_u32_noalloc(None, None, (1 << 24) + 1, None, None, 256, 0, None, None) == -1
    with pytest.raises(RuntimeError, match="tg_bin_count failed with code -1"):
        _lib.check(lib.tg_bin_count(None, 0, None, -1, 64, 64, 16, 16, None, None), "tg_bin_count", bits)


def test_python_entry_point_errors_without_gpu():
    """Error behaviour of reference src/trigrad/util.py:7-14 and wrapper.py:143-144."""
    import torch
    import trigrad_amd
    assert trigrad_amd.precision == torch.float32
    v = torch.zeros((3, 4)); i = torch.zeros((1, 3), dtype=torch.int32); c = torch.zeros((3, 3)); o = torch.zeros(3)
    with pytest.raises(TypeError, match="vertices must be on cuda, but got cpu"):
        trigrad_amd.render(v, i, c, o)
    with pytest.raises(ValueError, match="tile_width \\* tile_height must be <= 1024"):
        trigrad_amd.render(v, i, c, o, 64, 64, 33, 32)
    from trigrad_amd.util import create_check
    chk = create_check("cpu", torch.float32)
    chk(v, "v", (3, 4))
    with pytest.raises(ValueError, match="v must be of shape \\(3, 3\\)"):
        chk(v, "v", (3, 3))
    with pytest.raises(TypeError, match="v must be of type torch.float64"):
        chk(v, "v", (3, 4), torch.float64)
    chk(o, "o", 3)  # a bare int is promoted to a 1-tuple


def test_argument_errors_and_double_precision_do_not_need_the_torch_module(monkeypatch):
    """The C++ module for known frames is the float build's and the GPU's: what is refused for another reason says so where the
    module is not there, and double precision does without."""
    import torch
    import trigrad_amd
    from trigrad_amd import _C, _lib

    def missing(key_counts):
        raise AssertionError("the torch module was asked for")

    monkeypatch.setattr(_lib, "_torch_module", None)
    monkeypatch.setattr(_lib, "torch_module", missing)
    monkeypatch.setattr(_C, "_module_settings", None)
    v, i, c, o = torch.zeros((3, 4)), torch.zeros((1, 3), dtype=torch.int32), torch.zeros((3, 3)), torch.zeros(3)
    with pytest.raises(TypeError, match="vertices must be on cuda"):
        trigrad_amd.render(v, i, c, o, 16, 16)
    with pytest.raises(AttributeError):
        trigrad_amd.render([[0.0] * 4], i, c, o, 16, 16)
    _C.set_precision(torch.float64)
    try:
        with pytest.raises(TypeError, match="vertices must be on cuda"):
            trigrad_amd.render(v.double(), i, c.double(), o.double(), 16, 16)
    finally:
        _C.set_precision(torch.float32)


def test_product_does_not_reach_into_the_oracle():
    """Nothing under trigrad_amd/ may import, include or load the oracle."""
    for dirpath, _, files in os.walk(os.path.join(ROOT, "trigrad_amd")):
        for f in files:
            if f.endswith((".py", ".hip", ".hpp", ".h")):
                text = open(os.path.join(dirpath, f)).read()
                assert "oracle" not in text.lower(), f"{f} mentions the oracle"


def test_key_bits():
    from trigrad_amd import _C
    assert _C.key_bits(8160) == 45 and _C.key_bits(4096) == 44 and _C.key_bits(256) == 40 and _C.key_bits(1) == 33


def test_status_word_check_raises_without_a_gpu():
    """The check the frame makes of the list kernels' status word, on a host tensor."""
    import torch
    from trigrad_amd import _C
    _C.StatusCheck(torch.zeros((1,), dtype=torch.int32)).verify()
    bad = _C.StatusCheck(torch.tensor([1], dtype=torch.int32), what="tg_build_tile_lists")
    with pytest.raises(RuntimeError, match="tg_build_tile_lists: look-back wait timed out"):
        bad.verify()
    bad.verify()  # reported once
    _C._pending_checks.append(_C.StatusCheck(torch.tensor([1], dtype=torch.int32)))
    with pytest.raises(RuntimeError, match="look-back wait timed out"):
        _C.verify_finished_frames()
    _C.verify_finished_frames()
    assert _C._pending_checks == []


PAIRS_PROGRAM = r"""
#include <cstdio>
#include "tg_frame.hpp"
int main() {
    const uint32_t counted[2] = {700, 41}, expired[2] = {700, 42}, too_many[2] = {1025, 41};
    for (const uint32_t *word : {(const uint32_t *)nullptr, counted, expired, too_many})
        printf("%lld ", (long long)tg::FrameCount{word, 1024, 42}.pairs(33));
}
"""


def test_pairs_the_sort_takes(tmp_path):
    """How many pairs the sort's kernels take of a frame whose K is on the device, the rule compiled for the host: none where
    a wait of the scan expired (its K is a partial sum) or the buffers are too small."""
    import subprocess
    from trigrad_amd import build
    source, program = tmp_path / "pairs.hip", tmp_path / "pairs"
    source.write_text(PAIRS_PROGRAM)
    subprocess.run([os.environ.get("HIPCC", "/opt/rocm/bin/hipcc"), "--offload-host-only", "-std=c++17", "-w", "-I", build.CSRC,
                    str(source), "-o", str(program)], check=True)
    assert subprocess.run([str(program)], check=True, capture_output=True, text=True).stdout.split() == ["33", "700", "0", "0"]


def _device_compile(source, *flags):
    """Compiles one kernel file for the device with the build's flags; returns what the compiler said."""
    import subprocess
    from trigrad_amd import build
    return subprocess.run([os.environ.get("HIPCC", "/opt/rocm/bin/hipcc"), *[f for f in build.FLAGS if f != "-shared"],
                           "--offload-device-only", *flags, os.path.join(build.CSRC, source)], check=True, capture_output=True, text=True).stderr


def _assert_no_scratch_memory(source, kernels, flags, tmp_path):
    report = _device_compile(source, *flags, "-Rpass-analysis=kernel-resource-usage", "-c", "-o", str(tmp_path / "kernels.o"))
    names = re.findall(r"Function Name: (\S+)", report)
    scratch = re.findall(r"ScratchSize \[bytes/lane\]: (\d+)", report)
    assert len(names) == kernels == len(scratch)
    assert dict(zip(names, scratch)) == dict.fromkeys(names, "0")


@pytest.mark.parametrize("flags", [(), ("-DTG_DOUBLE_PRECISION",)])
def test_forward_kernels_need_no_scratch_memory(flags, tmp_path):
    """Scratch memory costs every launch of a kernel some microseconds: no instance of the forward kernels spills a register
    to it, in neither precision, by the compiler's own report."""
    _assert_no_scratch_memory("tg_forward.hip", 6, flags, tmp_path)


@pytest.mark.parametrize("flags", [(), ("-DTG_DOUBLE_PRECISION",)])
def test_backward_kernels_need_no_scratch_memory(flags, tmp_path):
    """The same of the backward kernels: three layouts each of the three compositors, two of them with and without a gradient of
    the depth map, and the split of the gradient blocks."""
    _assert_no_scratch_memory("tg_backward.hip", 16, flags, tmp_path)


@pytest.mark.parametrize("flags,scalar", [((), "float"), (("-DTG_DOUBLE_PRECISION",), "double")])
def test_record_parts_are_read_with_the_alignment_they_have(flags, scalar, tmp_path):
    """The parts of a record lie on scalar boundaries (y, z, w of a vertex; a triangle's indices and matrix): as written,
    before the optimiser narrows anything, no read of them promises more or goes beyond them."""
    _device_compile("tg_forward.hip", *flags, "-Xclang", "-disable-llvm-passes", "-emit-llvm", "-S", "-o", str(tmp_path / "forward.ll"))
    text = (tmp_path / "forward.ll").read_text()
    body = {name: re.search(r"define [^\n]*%s[^\n]*\n(.*?)\n}" % name, text, re.S).group(1)
            for name in ("DepthParts14fetch_vertices", "DepthParts12fetch_matrix")}
    reads = re.findall(r"load <(\d) x %s>, ptr \S+, align (\d+)" % scalar, "\n".join(body.values()))
    assert set(reads) <= {("4", "4")}  # the matrix: two fours and a scalar, packed
    assert body["DepthParts14fetch_vertices"].count("read_three") == 3 and body["DepthParts12fetch_matrix"].count("read_three") == 1
    copies = re.findall(r"define [^\n]*read_three[^\n]*\n.*?memcpy[^\n]* align (\d+) \S+ i64 (\d+)", text, re.S)
    size = 4 if scalar == "float" else 8
    assert sorted(copies) == sorted([("4", "12"), (str(size), str(3 * size))])


@pytest.mark.parametrize("columns,rows,slots_by_order", [(32, 24, (False, False)), (32, 32, (True, False)), (64, 32, (True, False)),
                                                         (65, 32, (True, True))])
def test_long_tiles_are_started_first_where_not_all_fit_at_once(columns, rows, slots_by_order):
    """768 workgroups of a per-pixel-order frame run at one time, 2048 of a tile-order one: only frames with more tiles keep
    slots for the tiles with long lists, 129 words and one a tile."""
    from trigrad_amd import _C
    tiles, counts = columns * rows, (3_000_000, 1_000_000)

    def scratch(pixel_order, n_triangles):
        return _C._FramePlan(counts[0], n_triangles, 16 * columns, 16 * rows, 16, 16, pixel_order, 32, 2_000_000, 0, 0.0).scratch_bytes

    slots = 768 + 256 * -(-4 * tiles // 256)
    for pixel_order, expected in zip((1, 0), slots_by_order):
        short = scratch(pixel_order, 1000)  # no list can be a long one
        assert scratch(pixel_order, counts[1]) - short == (slots if expected else 0)


@pytest.mark.parametrize("flags", [0, 1 | 4, 1 | 8, 1 | 4 | 16])
def test_buffers_for_a_rounded_number_of_triangles_serve_every_smaller_one(flags):
    """What frames with different numbers of triangles share is sized for the rounded number: nothing a frame needs is larger
    for a smaller one."""
    from trigrad_amd import _C
    assert [_C._round_count(n) for n in (1, 31, 32, 33, 1000, 65535, 65536, 65537, 2 ** 31 - 1)] == [
        1, 31, 32, 34, 1024, 65536, 65536, 69632, 2 ** 31 - 1]
    for n in (33, 500, 1023, 2047, 33_000, 65_000, 65_535, 65_537, 1_000_000):
        assert n <= _C._round_count(n) <= n + n // 16 + 1 and _C._round_count(_C._round_count(n)) == _C._round_count(n)
        for width, height, pixel_order in ((500, 400, 1), (1920, 1080, 1), (1920, 1080, 0)):
            sizes = [_C._FramePlan(0, k, width, height, 16, 16, pixel_order, k + 1, 300_000, flags, 0.0)
                     for k in (n, _C._round_count(n))]
            for field in ("kept_bytes", "scratch_bytes", "frame_bytes"):
                assert getattr(sizes[0], field) <= getattr(sizes[1], field)


@pytest.mark.parametrize("n_triangles,n_keys,tile,tile_order,pixel_order", [
    (20, 25, 16, 0, 1), (341, 450, 16, 0, 1), (300, 1499, 16, 0, 1), (300, 1500, 16, 8, 8), (300, 5999, 8, 0, 1), (300, 6000, 8, 8, 8)])
def test_a_gradient_block_for_each_xcd_by_the_keys_a_frame_has(n_triangles, n_keys, tile, tile_order, pixel_order):
    """Eight blocks where a triangle is in 20 waves on average, of the keys that were counted: the key buffers have room for
    more, a first frame's for 65536 more and those that an earlier frame's plan has for any number."""
    from trigrad_amd import _C, _lib
    for capacity in (_C._round_capacity(n_keys), 3 * n_triangles + 65536, 1 << 18):
        for per_pixel_sort, expected in ((0, tile_order), (1, pixel_order)):
            flags = _C._FRAME_BACKWARD | (_C._FRAME_ORDER_PLANES if per_pixel_sort else _C._FRAME_HIT_MASKS)
            frame = bytes(_C._FRAME_CALL.size) + _C._FRAME_RESULT.pack(n_keys, 1) + _C._FRAME_KIND.pack(
                3 * n_triangles, n_triangles, 256, 256, tile, tile, per_pixel_sort, 32, capacity, flags, 0, 0, 0.0)
            assert _lib.load(32).tg_frame_gradient_copies(frame) == expected


@pytest.mark.parametrize("flags,per_pixel_sort,expected", [(1, 1, 1), (1 | 2, 1, 8), (1 | 4, 1, 8), (1 | 4 | 16, 1, 8), (1, 0, 8), (1 | 8, 0, 8)])
def test_gradient_blocks_for_the_kernels_that_use_them(flags, per_pixel_sort, expected):
    """The backward kernel for frames without a saved blend order adds to the first block whatever its XCD: there is one."""
    from trigrad_amd import _C, _lib
    frame = bytes(_C._FRAME_CALL.size) + _C._FRAME_RESULT.pack(100_000, 1) + _C._FRAME_KIND.pack(
        3000, 1000, 256, 256, 16, 16, per_pixel_sort, 1001, 200_000, flags, 0, 0, 0.0)
    assert _lib.load(32).tg_frame_gradient_copies(frame) == expected


def test_backward_frame_takes_the_number_of_blocks_it_is_given():
    """The block is the caller's, who says how many (V,8) it holds: nothing that may have changed since it was allocated decides.
    A frame without vertices returns when its arguments are looked at."""
    from trigrad_amd import _C, _lib
    lib, somewhere = _lib.load(32), 1 << 20
    for per_pixel_sort in (0, 1):
        kind = _C._FramePlan(0, 100, 256, 256, 16, 16, per_pixel_sort, 32, 4096, _C._FRAME_BACKWARD, 0.0).kind
        for blocks, block, code in ((0, somewhere, 0), (1, somewhere, 0), (8, somewhere, 0), (8, somewhere + 4, -1), (1, 0, -1),
                                    (2, somewhere, -1), (7, somewhere, -1), (9, somewhere, -1), (-1, somewhere, -1), (8 + (1 << 32), somewhere, -1)):
            call = bytearray(_C._FRAME_BYTES)
            _C._FRAME_CALL.pack_into(call, 0, 0, 0, 0, 0, 0, 0, somewhere, 0, 0, 0, 0, 0, 0, _C._FRAME_GRADIENT_COPIES | blocks << 16, 0, 0, somewhere, block)
            _C._FRAME_RESULT.pack_into(call, _C._FRAME_CALL.size, 1 << 20, 1)
            call[-_C._FRAME_KIND.size:] = kind
            assert lib.tg_frame_backward((C.c_char * _C._FRAME_BYTES).from_buffer(call)) == code, (per_pixel_sort, blocks, block)


@pytest.mark.parametrize("missing", ["colors", "opacities"])
@pytest.mark.parametrize("phases", ["_FRAME_BIN", "all"])
def test_frames_with_records_are_refused_without_what_the_records_are_made_of(phases, missing):
    """The binning reads colours and opacities where it makes triangles' records: a null one of them is refused there, before
    anything is launched, and not found out by the kernel."""
    from trigrad_amd import _C, _lib
    lib, n, somewhere = _lib.load(32), 1_000_000, 1 << 20
    plan = _C._FramePlan(3 * n, n, 1920, 1080, 16, 16, 1, 32, 3_000_000, _C._FRAME_RECORDS, 0.0)
    call = bytearray(_C._FRAME_BYTES)
    host = (C.c_uint64 * 2)()  # four words
    phases = _C._FRAME_BIN if phases == "_FRAME_BIN" else _C._FRAME_BIN | _C._FRAME_LISTS | _C._FRAME_RASTER | _C._FRAME_WAIT
    _C._FRAME_CALL.pack_into(call, 0, somewhere, somewhere, 0 if missing == "colors" else somewhere, 0 if missing == "opacities" else somewhere,
                             somewhere, somewhere, somewhere, somewhere, somewhere, C.addressof(host), 0, 1,
                             plan.frame_bytes, phases, 0, 0, 0, 0)
    call[-_C._FRAME_KIND.size:] = plan.kind
    assert lib.tg_frame_has_records((C.c_char * _C._FRAME_BYTES).from_buffer(call))
    assert lib.tg_frame_forward((C.c_char * _C._FRAME_BYTES).from_buffer(call)) == -1
    assert b"null colors or opacities" in lib.tg_last_error()


def test_whether_a_frame_has_records_is_asked_of_any_frame():
    """A frame that the forward call refuses has none: a size of zero is no division, a null frame no read."""
    from trigrad_amd import _C, _lib
    lib, n = _lib.load(32), 1_000_000
    good = dict(n_vertices=3 * n, n_triangles=n, width=1920, height=1080, tile_w=16, tile_h=16, per_pixel_sort=1, max_layers=32, key_capacity=3_000_000)

    def has_records(**changed):
        kind = dict(good, **changed)
        return lib.tg_frame_has_records(bytes(_C._FRAME_CALL.size + _C._FRAME_RESULT.size) + _C._FRAME_KIND.pack(*kind.values(), _C._FRAME_RECORDS, 0, 0, 0.0))

    assert has_records() == 1 and lib.tg_frame_has_records(None) == 0
    for field in ("width", "height", "tile_w", "tile_h"):
        for size in (0, -1, -16, 1 << 40):
            assert has_records(**{field: size}) == 0
    assert has_records(key_capacity=1 << 30) == 0 and has_records(n_triangles=1 << 31, n_vertices=1 << 33) == 0


@pytest.mark.parametrize("n,keys_of_a_triangle,shown", [(499_999, 1.19, False), (500_000, 2.2, True), (524_288, 2.2, True), (524_289, 1.53, False),
                                                        (524_289, 1.19, True), (1_000_000, 2.2, False), (1_000_000, 1.53, False),
                                                        (1_690_000, 1.53, False), (1_700_000, 1.53, True), (1_700_000, 2.2, False), (2_000_000, 1.19, True)])
def test_shown_frames_in_tile_order_have_records_where_the_forward_pass_alone_gains_by_them(n, keys_of_a_triangle, shown):
    """In tile order the backward pass gains more by triangles' records than the forward pass, and a frame that is only shown has none:
    by its triangles and keys.  In per-pixel order, and where a backward pass follows, neither matters."""
    from trigrad_amd import _C, _lib
    lib, capacity = _lib.load(32), _C._round_capacity(int(n * keys_of_a_triangle))
    for per_pixel_sort, flags, expected in ((0, 0, shown), (0, _C._FRAME_BACKWARD | _C._FRAME_HIT_MASKS, n >= 500_000), (0, _C._FRAME_BACKWARD, n >= 500_000),
                                            (1, 0, True), (1, _C._FRAME_BACKWARD | _C._FRAME_ORDER_PLANES, True), (1, _C._FRAME_BACKWARD, False)):
        for records, n_vertices in ((1, 3 * n), (0, 3 * n), (1, 2 * n - 1)):
            kind = _C._FRAME_KIND.pack(n_vertices, n, 1920, 1080, 16, 16, per_pixel_sort, 32, capacity, flags | records * _C._FRAME_RECORDS, 0, 0, 0.0)
            assert lib.tg_frame_has_records(bytes(_C._FRAME_CALL.size + _C._FRAME_RESULT.size) + kind) == (expected and records and n_vertices == 3 * n)


@pytest.mark.parametrize("per_pixel_sort,flags", [(1, 0), (1, 1 | 2), (1, 1 | 4 | 16), (0, 0), (0, 1 | 8)])
def test_a_frame_without_records_keeps_no_room_for_them(per_pixel_sort, flags):
    """A record takes 128 bytes a triangle where a matrix takes 36: a mesh, and a frame of long lists in tile order, keep the matrices' place
    only, and the plan that later frames share has the room if, and only if, one of them may have records."""
    from types import SimpleNamespace
    from unittest import mock
    from trigrad_amd import _C, _lib
    left = {}
    module = SimpleNamespace(remember=lambda key, kind, frame_bytes, low, high: left.update({key: kind}), state_bytes=lambda *_: 1 << 60)

    def kept(n_vertices, n, capacity=3_000_000, records=_C._FRAME_RECORDS):
        return _C._FramePlan(n_vertices, n, 1920, 1080, 16, 16, per_pixel_sort, 32, capacity, flags | records, 0.0).kept_bytes

    def left_for(n_vertices, n):
        left.clear()
        with mock.patch.object(_C, "_module", lambda: module):
            _C._leave_plan((n_vertices, n, 1920, 1080, 16, 16, per_pixel_sort, 32, 3_000_000, flags, 0.0), bool(flags & 1), SimpleNamespace(index=0), 0)
        return list(left.items())

    for n in (149_999, 150_000, 155_648, 499_999, 524_288, 524_289, 1_000_000, 1_300_000):
        n_rounded, least = _C._round_count(n), 150_000 if per_pixel_sort else 500_000
        assert kept(2 * n - 1, n) == kept(n // 2, n) == kept(3 * n, n, records=0)
        assert round((kept(2 * n, n) - kept(n, n)) / n, 2) == (92 if n >= least else 0)
        if not per_pixel_sort:
            assert kept(3 * n, n, 8_000_000) == kept(3 * n, n, 8_000_000, records=0)
        keys = set()
        for n_vertices in (n // 2, 2 * n - 1, 2 * n, 3 * n):
            (key, kind), = left_for(n_vertices, n)
            keys.add(key)
            of_plan = _C._FRAME_KIND.unpack(kind)[10]
            assert of_plan >= kept(n_vertices, n)
            assert of_plan == kept(0 if n_vertices < 2 * n else 3 * n_rounded, n_rounded)
        assert len(keys) == 2
    assert not left_for(0x7fffffff, (1 << 30) - 1) and len(left_for(0x7fffffff, 1 << 30)) == 1


@pytest.mark.parametrize("few,many", [(1, 2049), (2048, 1 << 24), ((1 << 24) + 1, (1 << 25) + 1)])
def test_state_words_of_the_frame_scan_keep_their_place(few, many):
    """What calls share in a frame state must lie where no call puts anything else, whatever its number of triangles: with more
    triangles the state grows by what a triangle takes behind it (4 bytes of offset, 48 of record), and by nothing else."""
    from trigrad_amd import _lib
    lib = _lib.load(32)
    grown = lib.tg_bin_frame_workspace_bytes(many, 1000, 640, 480, 16, 16) - lib.tg_bin_frame_workspace_bytes(few, 1000, 640, 480, 16, 16)
    up = lambda n: -(-n // 256) * 256
    assert grown == up(4 * many) - up(4 * few) + up(48 * many) - up(48 * few)
