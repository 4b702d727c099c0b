"""The autotuner's candidates: each launches something else, or it could only tell noise apart."""
import importlib

at = importlib.import_module("wgpu-sigops_amd.autotune")


def test_candidates_differ():
    knobs = {"waves", "tile_rounds", "bucket_order"}  # what the mixed batch's launch depends on
    assert at.DEFAULT in at.CANDIDATES
    seen = [tuple(sorted((k, v) for k, v in c.items() if k in knobs)) for c in at.CANDIDATES]
    assert len(set(seen)) == len(at.CANDIDATES)
