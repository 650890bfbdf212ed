"""Launch plans of the dense encoding, on the CPU.

A workgroup searches at most ``pairs_per_block`` (sample, feature) pairs at a
time; a block of its samples must never hold more, whatever the features and
bins, or the pairs beyond would be left out of the output.
"""

from __future__ import annotations

import pytest

from piecewiselinearembeddings_optimized_amd import capi

FEATURES = (1, 2, 7, 64, 300, 1021, 1024, 2043, 2044, 2045, 2046, 2047, 2048, 2049, 2200, 2201, 2300, 2408, 2409)
WIDER = (2410, 2630, 3683, 3684, 4096, 5000, 20001, 100000)      # the backward takes these too
BINS = (1, 2, 3, 4, 16, 48, 100, 256, 1000, 4000, 9001)
SAMPLES = (1, 16, 255, 1000, 4080, 4096, 4200, 16384, 300000)


@pytest.mark.parametrize("backward", [False, True], ids=["forward", "backward"])
@pytest.mark.parametrize("bins", BINS)
def test_block_holds_no_more_pairs_than_are_searched(bins, backward):
    for f in FEATURES + (WIDER if backward else ()):
        if f * (bins + 1) > (2**31 - 1) // 2 // 2:
            continue
        for n in SAMPLES:
            for total in {f * bins, (f * bins + 3) // 4 * 4, max(f * bins // 2, 1)}:
                pl = capi.encode_plan(n, f, bins, total, backward)
                if pl["groups"] == 0:
                    continue        # whole rows, or one thread per pair
                assert pl["rows_per_block"] >= 1 and pl["chunks"] >= 1
                assert pl["rows_per_block"] * pl["features_searched"] <= pl["pairs_per_block"], (n, f, total, pl)
                assert pl["features_per_group"] * pl["groups"] >= f
                assert pl["lds_bytes"] <= 160 * 1024


def test_forward_feature_limit():
    assert capi.encode_plan(8, 2409, 1, 2409)["groups"] >= 1
    assert capi.encode_plan(4096, 2409, 4000, 2409 * 4000)["groups"] == 0     # whole rows: all in LDS
    with pytest.raises(capi.PleError):
        capi.encode_plan(8, 2410, 1, 2410)
    assert capi.encode_plan(300000, 2410, 1, 2410, backward=True)["groups"] >= 1
