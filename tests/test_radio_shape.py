"""Launch shapes of the radio projection, computed on the host: what the knobs of
set_tuning select. A small library around shape_projection, linked to the product library,
is compiled for the test."""
import ctypes
import os
import subprocess

import pytest

import c8mi

PACKAGE = os.path.dirname(os.path.dirname(os.path.abspath(c8mi.__file__)))

SOURCE = r"""
#include <stdexcept>
#include "radio/radio_launch.hpp"
using namespace c8mi::radio;
// shape: tile bins, window tiles, observers per workgroup, threads, tracks per chunk, chunks
extern "C" int shape(int coreas, int zhs, int fast, unsigned observers, unsigned long bins, unsigned long count,
                     int tuned, unsigned long chunk, unsigned tile, unsigned target, unsigned threads,
                     unsigned long* out) {
  try {
    ProjectionLaunch L{};
    LaunchTuning tuning;
    if (tuned) tuning = make_tuning(chunk, tile, target, threads);
    shape_projection(L, coreas, zhs, fast, observers, bins, count, tuning);
    unsigned long const values[6] = {L.tile_bins, L.bin_tiles, L.group, L.block_threads, L.chunk_size, L.chunks};
    for (int k = 0; k < 6; ++k) out[k] = values[k];
    return 0;
  } catch (std::invalid_argument const&) {
    return 1;
  } catch (std::length_error const&) {
    return 2;
  }
}
// the tracks of `count` that a tuned CoREAS launch takes
extern "C" unsigned long taken(unsigned observers, unsigned long bins, unsigned long count, unsigned long chunk,
                               unsigned tile) {
  LaunchTuning const tuning = make_tuning(chunk, tile, 0, 0);
  return launchable(count, [&](std::uint64_t tracks) {
    ProjectionLaunch L{};
    shape_projection(L, true, false, true, observers, bins, tracks, tuning);
  });
}
"""


@pytest.fixture(scope="module")
def shape(tmp_path_factory):
    folder = tmp_path_factory.mktemp("shape")
    source, library = folder / "shape.cpp", folder / "libshape.so"
    source.write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I" + os.path.join(PACKAGE, "csrc"), "-I" + os.path.join(os.path.dirname(PACKAGE), "include"),
                    str(source), "-o", str(library), "-L" + PACKAGE, "-lc8mi", "-Wl,-rpath," + PACKAGE], check=True)
    lib = ctypes.CDLL(str(library))

    def call(fast, observers, bins, count, coreas=True, zhs=False, tuning=None):
        out = (ctypes.c_ulong * 6)()
        t = tuning or {}
        status = lib.shape(int(coreas), int(zhs), int(fast), ctypes.c_uint(observers), ctypes.c_ulong(bins),
                           ctypes.c_ulong(count), int(tuning is not None), ctypes.c_ulong(t.get("chunk_tracks", 0)),
                           ctypes.c_uint(t.get("tile_bins", 0)), ctypes.c_uint(t.get("target_workgroups", 0)),
                           ctypes.c_uint(t.get("block_threads", 0)), out)
        if status:
            return status
        return dict(zip(("tile_bins", "bin_tiles", "group", "threads", "chunk", "chunks"), out))

    call.library = lib
    return call


SIZES = [(160, 2048, 1 << 20), (160, 1024, 30000), (24, 512, 1500), (7, 300, 200000), (64, 4096, 100003)]


@pytest.mark.parametrize("observers,bins,count", SIZES)
@pytest.mark.parametrize("coreas,zhs", [(True, False), (False, True), (True, True)])
def test_knobs_left_automatic_keep_the_estimate(shape, observers, bins, count, coreas, zhs):
    """set_tuning() with defaults, or with split alone (no part of the shape), is no tuning."""
    plain = shape(True, observers, bins, count, coreas, zhs)
    assert shape(True, observers, bins, count, coreas, zhs, tuning={}) == plain
    if coreas and zhs:  # the fused launch is not estimated
        assert (plain["group"], plain["threads"]) == (1, 256)
    elif count == 1 << 20:
        assert plain["group"] > 1 and plain["threads"] == 1024
    exact = shape(False, observers, bins, count, coreas, zhs)
    assert shape(False, observers, bins, count, coreas, zhs, tuning={}) == exact
    assert (exact["group"], exact["threads"]) == (1, 512)


@pytest.mark.parametrize("observers,bins,count", SIZES)
@pytest.mark.parametrize("tuning", [dict(target_workgroups=4096), dict(chunk_tracks=2048), dict(tile_bins=100),
                                    dict(block_threads=256), dict(chunk_tracks=1024, block_threads=1024)])
def test_a_knob_selects_one_observer_a_workgroup(shape, observers, bins, count, tuning):
    got = shape(True, observers, bins, count, tuning=tuning)
    assert got["group"] == 1
    assert got["threads"] == tuning.get("block_threads", 512)
    if "chunk_tracks" in tuning:
        assert got["chunk"] == tuning["chunk_tracks"]
    if "tile_bins" in tuning:
        assert got["tile_bins"] == 100
    if "target_workgroups" in tuning:
        chunks = max(8, min(4096 // (observers * got["bin_tiles"]), count // 32768) // 8 * 8)
        assert got["chunks"] <= chunks


def test_refused_knobs(shape):
    assert shape(True, 10, 100, 1000, tuning=dict(block_threads=128)) == 1
    assert shape(True, 10, 100, 1000, tuning=dict(chunk_tracks=100)) == 1
    assert shape(True, 10, 100, 1000, tuning=dict(chunk_tracks=512, block_threads=1024)) == 1
    assert shape(True, 4096, 1 << 20, 1 << 24, tuning=dict(chunk_tracks=256, tile_bins=1)) == 2


def test_a_list_too_large_for_one_launch(shape):
    """A batch of fronts is projected in launches that 2^32 workgroups hold."""
    taken = shape.library.taken
    taken.restype = ctypes.c_ulong
    n = lambda count, tile: taken(ctypes.c_uint(160), ctypes.c_ulong(65536), ctypes.c_ulong(count), ctypes.c_ulong(256),
                                  ctypes.c_uint(tile))
    per_chunk = 160 * 65536
    got = n(1 << 20, 1)
    assert got == 1 << 16 and got // 256 * per_chunk < 1 << 32 <= 2 * got // 256 * per_chunk
    assert n(100000, 1) == 100000
    assert n(1 << 20, 1000) == 1 << 20
