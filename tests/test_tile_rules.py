"""The kernels' rules on the CPU: the tiles a wave leaves out, the form of the
16-bit backward that a scale takes, the form of the forward that a grid takes.

`tile_unseen` (graph-kernel-injection_amd/csrc/gki_common.cuh) must never hold
for a tile of which some row sees a key under the oracle's token rule, and
holds whenever no in-range row sees one (else work would be done for nothing).
"""

from __future__ import annotations

import math
import os
import shutil
import subprocess

import numpy as np
import pytest

from oracle import streaming_oracle as so

HERE = os.path.dirname(os.path.abspath(__file__))
REPO = os.path.dirname(HERE)
CSRC = os.path.join(REPO, "graph-kernel-injection_amd", "csrc")
TILE = 64


@pytest.fixture(scope="module")
def rules_exe(tmp_path_factory):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not available")
    exe = str(tmp_path_factory.mktemp("tile_rules") / "tile_rules_host")
    subprocess.run([hipcc, "--offload-arch=gfx950", "-O1", "-std=c++17", f"-I{CSRC}",
                    f"-I{os.path.join(REPO, 'include')}", os.path.join(HERE, "tile_rules_host.hip"),
                    "-o", exe], check=True, capture_output=True, timeout=600)
    return exe


def _run(exe, what, lines):
    return subprocess.run([exe, what], input="\n".join(lines) + "\n", capture_output=True, text=True, check=True,
                          timeout=120).stdout.split()


PLAIN, ROW, PRE = 0, 1, 2
FP32, FP16, BF16 = 0, 1, 2


def test_an_operand_of_the_backward_carries_exact_scales_only(rules_exe):
    """The powers of two 2^-4 .. 1, of either sign; elsewhere dS is scaled in fp32."""
    scales = [0.0] + [s * m * 2.0**e for e in range(-40, 40) for m in (1.0, math.sqrt(2), 1.999) for s in (1, -1)]
    for dtype in (FP32, FP16, BF16):
        out = _run(rules_exe, "form", [f"{dtype} {s!r}" for s in scales])
        assert len(out) == len(scales)
        for s, form in zip(scales, map(int, out)):
            mag = abs(float(np.float32(s)))
            if dtype == FP32 or 0 < mag < 2.0**-30 or mag >= 2.0**30:
                want = PLAIN
            else:
                want = PRE if 2.0**-4 <= mag <= 1 and math.frexp(mag)[0] == 0.5 else ROW
            assert form == want, (dtype, s, form)


def test_kv_tiles_of_a_row_are_bounded(rules_exe):
    """row_kv_tiles: never less than the longest list of the token rule, at most one
    (an unaligned window) and the sinks' tiles above it in the middle of a long row."""
    rng = np.random.default_rng(3)
    cases = [(int(rng.integers(1, 700)), int(rng.integers(1, 900)), int(rng.choice([0, 1, 4, 100])),
              int(rng.choice([0, 1, 31, 64, 200, 2**31 - 1])), rows) for _ in range(100) for rows in (64, 128)]
    out = _run(rules_exe, "grid", [f"64 1 {n_q} {n_kv} 1 {s} {w} {rows}" for n_q, n_kv, s, w, rows in cases])
    for (n_q, n_kv, sink, window, rows), got in zip(cases, map(int, out[::4])):
        tiles = so.tile_classes(np.ones((-(-n_q // 64), -(-n_kv // 64)), np.int32), n_q, n_kv, 64, 64, rows, TILE, True,
                                sink, min(window, n_q + n_kv))
        longest = int((tiles != 0).sum(1).max())
        assert longest <= got <= -(-n_kv // TILE)
        if n_q < n_kv // 3 and n_q % rows == 0 and window < n_kv // 3:
            assert got <= longest + 1 + -(-sink // TILE)
    assert _run(rules_exe, "grid", ["64 1 100 1000 0 0 0 64", "64 1 9 64 0 0 0 64"])[::4] == ["8", "1"]


def test_grids_whose_tiles_share_their_keys(rules_exe):
    """Two workgroups of shares per tile while all run at once (128 tiles); up to 256
    tiles of long lists where a CU holds two; head_dim 128 never past one per CU."""
    def lines(d, tiles, n_kv, window, causal=1):
        return f"{d} {tiles} 128 {n_kv} {causal} 4 {window} 128"

    got = {}
    cases = [(d, tiles, n_kv, window) for d in (16, 32, 64, 128) for tiles in (1, 128, 129, 256, 257, 4096)
             for n_kv, window in ((64, 64), (1024, 64), (1024, 256), (1024, 400), (9000, 2048))]
    for case, form in zip(cases, _run(rules_exe, "grid", [lines(*c) for c in cases])[1::4]):
        got[case] = form == "1"
    for (d, tiles, n_kv, window), split in got.items():
        assert split == (tiles <= 128 or (d <= 64 and tiles <= 256 and window >= 256)), (d, tiles, n_kv, window)


def test_fp32_blocks_per_workgroup(rules_exe):
    """Four, two, one workgroups per tile or item while they fit the card, fewer for
    the wider heads; one from 129 tiles on where a row sees one or two kv tiles."""
    def blocks(d, n, n_kv=9000):
        out = _run(rules_exe, "grid", [f"{d} {n} 64 {n_kv} 1 4 2048 64"])
        return int(out[2]), int(out[3])

    for d, one, k_one, k_two in ((16, 256, 128, 384), (32, 256, 128, 384), (64, 128, 64, 256), (128, 64, 0, 128)):
        for n in (1, 64, 65, 128, 129, 256, 257, 384, 385, 512, 100000):
            rows, kv = blocks(d, n)
            assert rows == (1 if n <= one else 2 if n <= 384 else 4), (d, n)
            assert kv == (1 if n <= k_one else 2 if n <= k_two else 4), (d, n)
            assert blocks(d, n, 128)[0] == (4 if n > 128 else rows), (d, n)


def test_unseen_tiles_are_exactly_those_without_a_visible_key(rules_exe):
    rng = np.random.default_rng(5)
    lines, want = [], []
    for _ in range(150):
        n_kv = int(rng.integers(1, 500))
        n_q = int(rng.integers(1, 600))
        causal = bool(rng.random() < 0.85)
        sink = int(rng.choice([0, 1, 4, 64, 100]))
        window = int(rng.choice([0, 1, 31, 64, 100, 700, 2**31 - 1]))
        vis = so.token_mask(n_q, n_kv, sink, min(window, n_q + n_kv + 1)) if causal else np.ones((n_q, n_kv), bool)
        for q_lo in range(0, n_q, 32):
            for k0, n_k in [(k, n) for n in (TILE, TILE // 2) for k in range(0, n_kv, n)]:
                lines.append(f"{n_q} {n_kv} {int(causal)} {sink} {window} {q_lo} {q_lo + 31} {k0} {n_k}")
                want.append((not causal, bool(vis[q_lo:q_lo + 32, k0:k0 + n_k].any()), q_lo + 32 <= n_q))
    out = _run(rules_exe, "unseen", lines)
    assert len(out) == len(want)
    skipped = 0
    for line, got, (never, seen, whole) in zip(lines, out, want):
        unseen = got == "1"
        assert not (unseen and (seen or never)), line
        # and no visited tile is for nothing, where every row exists (past the sinks; a window of 0 sees only those)
        sink, window, k0 = (int(line.split()[i]) for i in (3, 4, 7))
        if whole and not never and not seen and k0 >= sink and window > 0:
            assert unseen, line
        skipped += unseen
    assert skipped > 1000
