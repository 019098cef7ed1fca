"""Differential attention: a group of waves per softmax branch, in workgroups of 64 and 128 rows, or the branches one after the other
(plan_diff in csrc/api.hip), against fp64 at the edges of the tiles."""
import ctypes as C
import os
import subprocess
import sys
from pathlib import Path

import pytest
import torch

from flashlight_amd import _ffi
from tests.test_abi import good_params

DEV = "cuda"
NONE, CAUSAL, SLIDING, PREFIX = _ffi.MASK_NONE, _ffi.MASK_CAUSAL, _ffi.MASK_SLIDING, _ffi.MASK_PREFIX_LM


def _shape(B, H, S, D, mask):
    """(rows per workgroup, keys per tile, groups of waves) the library plans."""
    p = good_params(B=B, Hq=H, Hkv=H, L=S, D=D, Dv=128)
    p.diff, p.mask_kind, p.window, p.prefix = 1, mask, 100, 100
    out = (C.c_int64 * 8)()
    assert _ffi.load_library().fl_attn_plan(C.byref(p), out) == 0, _ffi.last_error()
    assert out[4] <= 160 * 1024
    return out[0], out[1], out[7]


def test_which_calls_take_which_workgroups():
    assert _shape(2, 16, 4096, 64, CAUSAL) == (128, 64, 2) and _shape(2, 16, 1000, 64, CAUSAL) == (64, 64, 2)
    assert _shape(6, 8, 2048, 64, CAUSAL) == (64, 64, 2) and _shape(6, 8, 2048, 64, NONE) == (128, 64, 2)
    assert _shape(1, 2, 1000, 64, CAUSAL) == (128, 32, 2) and _shape(1, 2, 1100, 64, CAUSAL) == (64, 64, 2)
    assert _shape(16, 16, 200, 64, NONE) == (128, 32, 1) and _shape(16, 16, 200, 64, CAUSAL) == (64, 64, 2)
    assert _shape(4, 16, 4096, 64, SLIDING) == (64, 64, 2) and _shape(4, 16, 4096, 128, SLIDING) == (128, 32, 1)
    assert _shape(16, 16, 256, 128, CAUSAL) == (128, 32, 1) and _shape(2, 16, 1000, 128, CAUSAL) == (128, 64, 2)


def test_short_walks_of_many_workgroups():
    """Where two workgroups of 128 rows per compute unit are ahead of a group per branch."""
    turns = (128, 32, 1)  # one branch after the other
    for mask in (NONE, CAUSAL, PREFIX):
        assert _shape(33, 32, 130, 128, mask) == turns and _shape(50, 16, 200, 128, mask) == turns and _shape(5, 16, 200, 128, mask) == (128, 64, 2)
        assert _shape(5, 16, 1500, 128, mask) == (128, 64, 2)
    assert _shape(20, 16, 600, 128, NONE) == turns and _shape(8, 16, 600, 128, NONE) == (128, 64, 2) and _shape(20, 16, 600, 128, CAUSAL) == (128, 64, 2)
    assert _shape(1, 75, 450, 128, CAUSAL) == turns and _shape(1, 72, 450, 128, CAUSAL) == (128, 64, 2)
    assert _shape(1, 251, 850, 128, PREFIX) == turns and _shape(1, 101, 850, 128, PREFIX) == (128, 64, 2)
    assert _shape(1, 651, 200, 64, NONE) == turns and _shape(1, 448, 200, 64, NONE) == turns and _shape(1, 320, 256, 64, NONE) == (64, 64, 2)
    assert _shape(1, 325, 512, 64, NONE) == turns and _shape(1, 325, 420, 64, NONE) == (64, 64, 2) and _shape(1, 325, 512, 64, CAUSAL) == (64, 64, 2)
    assert _shape(1, 103, 600, 64, NONE) == (64, 64, 2) and _shape(1, 96, 600, 64, NONE) == turns


@pytest.mark.parametrize("tile,shapes", [
    # tiles without a form for the branches one after the other take a group for each, also where the rule prefers one group ...
    ("32x64x4x2", {(4, 16, 4096, 128, SLIDING): (128, 64, 2), (16, 16, 200, 64, NONE): (128, 64, 2)}),
    ("32x64x2x2", {(16, 16, 200, 64, NONE): (64, 64, 2)}),
    # ... and the 32-key tile of head dim 128 has no form with two
    ("32x32x4x2", {(2, 16, 1000, 128, CAUSAL): (128, 32, 1), (16, 16, 200, 64, NONE): (128, 32, 1), (2, 16, 1000, 64, CAUSAL): (128, 32, 2)}),
])
def test_a_forced_tile_is_planned_with_groups_that_it_has(tile, shapes):
    # (the knob is read once per process)
    script = "from tests.test_differential_branches import _shape\nprint([_shape(*s) for s in %r])" % (list(shapes),)
    env = dict(os.environ, FL_TILE=tile)
    got = subprocess.run([sys.executable, "-c", script], env=env, cwd=Path(__file__).parent.parent, capture_output=True, text=True, timeout=300)
    assert got.returncode == 0, got.stderr
    assert got.stdout.splitlines()[-1] == str(list(shapes.values()))


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("B,H,Hkv,Lq,Lk", [(1, 2, 1, 33, 33), (3, 6, 3, 129, 129), (3, 7, 7, 191, 191), (2, 9, 9, 257, 257), (1, 18, 6, 65, 321),
                                           (1, 17, 17, 300, 64), (16, 32, 32, 100, 100), (29, 4, 2, 511, 511), (1, 3, 3, 1025, 1025)])
def test_results_against_fp64(B, H, Hkv, Lq, Lk, D, dtype):
    g = torch.Generator().manual_seed(Lq + Lk + D)
    mk = lambda *s: torch.randn(*s, generator=g).to(dtype).to(DEV)  # noqa: E731
    q, k, v = mk(B, 2 * H, Lq, D), mk(B, 2 * Hkv, Lk, D), mk(B, Hkv, Lk, 128)
    wide = lambda t: t.double().repeat_interleave(H // Hkv, dim=1)  # noqa: E731
    diff = torch.arange(Lk, device=DEV)[None] - torch.arange(Lq, device=DEV)[:, None]
    keep = {NONE: diff == diff, CAUSAL: diff <= 0, SLIDING: (diff <= 0) & (diff >= -70), PREFIX: (diff <= 0) | (torch.arange(Lk, device=DEV) < 40)[None]}
    vd = wide(v)
    for mask, attended in keep.items():
        if mask in (SLIDING, PREFIX) and Lq != Lk:
            continue  # (refused)
        out = _ffi.attn_fwd(q, k, v, mask_kind=mask, window=70, prefix=40, diff=True, lambda_full=0.7)
        ref, bound = 0.0, 0.0
        # Each branch: weights rounded to 16 bits (u of their size; fp16 weights far below the reference are subnormal, together less than
        # 2^-15 of the row's sum), numerator and row sum alike; then one rounding of the result.
        u = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
        for br, factor in ((0, 1.0), (1, -0.7)):
            qb, kb = q[:, br * H:(br + 1) * H].double(), wide(k[:, br * Hkv:(br + 1) * Hkv])
            s = (torch.matmul(qb, kb.transpose(-1, -2).contiguous()) * D ** -0.5).masked_fill(~attended, float("-inf"))
            w = torch.softmax(s, -1).nan_to_num()  # (a row that attends nothing gives zeros)
            o = torch.matmul(w, vd)
            ref = ref + factor * o
            bound = bound + abs(factor) * (u * (torch.matmul(w, vd.abs()) + o.abs()) + 2.0 ** -15 * v.abs().max().item())
        assert torch.isfinite(out).all(), mask
        assert ((out.double() - ref).abs() <= bound + u * ref.abs()).all(), mask
