"""Which form a forward call takes (key groups, split keys), at sizes where the
other forms measured slower: each case names the time of every form in us."""

import pytest
import torch

from mlx_primitives import _native

BF, F32 = torch.bfloat16, torch.float32


def form(B, H, Sq, Sk, D, causal, dtype=BF, left=-1, right=-1, page=0, alibi=False):
    if causal and Sk > Sq and not page:
        causal, right = False, Sk - Sq
    groups, splits, _ = _native.fwd_form(B, H, Sq, Sk, D, causal, left, right, dtype, page, alibi)
    return groups, splits > 1


@pytest.mark.parametrize("args,want", [
    # one tile of keys: cutting it only adds the merge (1 / 2 / 4 groups)
    (dict(B=6, H=2, Sq=66, Sk=66, D=128, causal=False), (1, False)),      # 9.0 / 9.3 / 10.6
    (dict(B=1, H=1, Sq=98, Sk=98, D=128, causal=False), (1, False)),      # 9.1 / 9.5 / 10.3
    (dict(B=3, H=7, Sq=39, Sk=39, D=128, causal=False, left=10, right=10), (1, False)),  # 8.6 / 8.4 / 9.6
    # one round of workgroups against more of them
    (dict(B=1, H=88, Sq=162, Sk=162, D=64, causal=True), (2, False)),     # 9.6 / 7.8 / 11.9
    (dict(B=1, H=17, Sq=3689, Sk=3689, D=64, causal=True), (1, False)),   # 57.7 / 67.3 / 64.5
    (dict(B=4, H=7, Sq=4431, Sk=4431, D=64, causal=False), (1, False)),   # 152.9 / 182.9 / 245.9
    (dict(B=3, H=20, Sq=563, Sk=563, D=64, causal=True, left=20), (1, False)),  # 13.7 / 16.4 / 20.1
    (dict(B=2, H=16, Sq=2048, Sk=2048, D=128, causal=True), (2, False)),  # 55.4 / 47.6 / 72.4
    # pages in 64-key tiles: two groups save little of a step
    (dict(B=3, H=12, Sq=3569, Sk=3584, D=64, causal=False, page=16), (1, False)),
    # float32: a split and its merge (1, split / 2, split / 2)
    (dict(B=1, H=11, Sq=62, Sk=838, D=32, causal=False, dtype=F32), (2, True)),  # 18.9 / 13.9 / 25.2
    (dict(B=7, H=3, Sq=55, Sk=795, D=32, causal=True, dtype=F32), (2, True)),    # 19.2 / 14.0 / 24.3
    (dict(B=1, H=4, Sq=1093, Sk=1093, D=32, causal=False, dtype=F32), (2, True)),  # 20.5 with one group
])
def test_form(args, want):
    assert form(**args) == want
