"""Which kernels a prefill product launches, on a HIP runtime without a device
(tests/host_checks)."""
import subprocess

import pytest

from test_host_failures import checks  # noqa: F401  (the fixture)


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
    (m, *s) for m in ("q4", "q8", "bf16")
    for s in ((0, 64, 256), (0, 256, 512), (0, 512, 512), (1, 1024, 256), (1, 2048, 512))
    if (m, s) != ("bf16", (1, 2048, 512))])
def test_small_products_are_one_launch(checks, mode, pair, N, K):
    most = {"q4": (48, 40), "q8": (48, 48), "bf16": (32, 16)}[mode][pair]
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
