"""Which kernels a prefill product launches, on a HIP runtime without a device
(tests/host_checks)."""
import os
import subprocess

import pytest

from test_gpu_prefill import STREAM_CUTS, TILE_SHAPES
from test_host_failures import checks  # noqa: F401  (the fixture)

MODES = ("q4", "q8", "bf16")
# most tokens of a streamed product and of a streamed gate/up pair
STREAMED = {"q4": (48, 40), "q8": (48, 48), "bf16": (32, 16)}


def launches(checks, products, env=None):
    """Per product (mode, pair, T, N, K[, bytes off 16]) its launches: (name, grid, block, lds)."""
    exe, folder = checks
    lines = "".join("%s %d %d %d %d %d\n" % (p if len(p) == 6 else p + (0,)) for p in products)
    r = subprocess.run([exe, folder, "launches"], input=lines, env=env, capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stderr
    out = []
    for line in r.stdout.splitlines():
        assert not line.startswith("error"), line
        f = [e.split() for e in line.split("\t") if e]
        out.append([(e[0], tuple(map(int, e[1:4])), int(e[4]), int(e[5])) for e in f])
    assert len(out) == len(products)
    return out


# A product of few blocks is one slice: its planes' sum would be a launch of its
# own, which takes longer than the rest (a bf16 pair of 2048 x 512 takes the same
# time either way).
@pytest.mark.parametrize("mode,pair,N,K", [
    (m, *s) for m in MODES
    for s in ((0, 64, 256), (0, 256, 512), (0, 512, 512), (1, 1024, 256), (1, 2048, 512))
    if (m, s) != ("bf16", (1, 2048, 512))])
def test_small_products_are_one_launch(checks, mode, pair, N, K):
    most = STREAMED[mode][pair]
    for T, calls in zip((2, 8, 16, most), launches(checks, [(mode, pair, T, N, K) for T in (2, 8, 16, most)])):
        assert len(calls) == 1 and calls[0][1][2] == 1, (T, calls)


# The 64 x 128 tile fits a CU twice with Q4 and bf16 weights, not with Q8 ones: 352
# workgroups of an unsplit gate/up are one and a half rounds or two.  A grid's LDS
# is that of the layout the kernel is compiled with (csrc/common/wide_lds.h).
@pytest.mark.parametrize("mode,lds", [("q4", 5 * 8192 + 3 * 10240 + 1024), ("q8", 5 * 8192 + 3 * 18432 + 1024),
                                      ("bf16", 5 * (8192 + 8192))])
def test_wide_tile_residency(checks, mode, lds):
    wide = [c for c in launches(checks, [(mode, 1, 64, 11264, 6144)])[0] if "wgateup" in c[0]]
    assert [c[0] for c in wide] == ["gh_pf_wgateup_%s_m1_n128_k" % mode] and wide[0][3] == lds
    assert (2 * lds <= 160 * 1024) == (mode != "q8")


# The shapes of test_gpu_prefill.py reach the kernels they are there for.
@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("shape", TILE_SHAPES, ids=lambda s: "-".join(map(str, s[:4])))
def test_tile_shapes_reach_their_kernels(checks, mode, shape):
    want = shape[4] if mode == "q4" else shape[5] or shape[4]
    op, form = want.split("_", 1)
    names = [c[0] for c in launches(checks, [(mode, *shape[:4])])[0]]
    assert "gh_pf_%s_%s_%s" % (op, mode, form) in names, names


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("T,N,K,cut", STREAM_CUTS)
def test_forced_cuts_are_taken(checks, mode, T, N, K, cut):
    kr, rgw, nw = map(int, cut.split(","))
    for pair in (0, 1):
        call = launches(checks, [(mode, pair, T, N, K)], dict(os.environ, GH_PF_STREAM=cut))[0]
        streamed = [c for c in call if c[0].startswith(("gh_pf_sgemm_", "gh_pf_sgateup_"))]
        assert bool(streamed) == (T <= STREAMED[mode][pair]), call
        if streamed:
            grid = (-(-(-(-N // 16)) // (nw * rgw)), 1, -(-K // 32 // kr))
            assert streamed[0][1:3] == (grid, 64 * nw), (streamed, grid)


# Weights off 16 bytes, and columns off 128, take the tile GEMM; all else does not.
@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("pair", [0, 1])
def test_what_the_tile_gemm_serves(checks, mode, pair):
    for T in (1, 16, 17, 48, 49, 200, 512):
        for K, off in ((3840, 0), (3872, 0)) + (((3840, 4),) if mode != "bf16" else ()):
            tile = [c for c in launches(checks, [(mode, pair, T, 2048, K, off)])[0]
                    if c[0].startswith(("gh_pf_gemm_", "gh_pf_gateup_"))]
            assert bool(tile) == (K % 128 != 0 or off != 0), (T, K, off)
