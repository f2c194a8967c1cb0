"""Which window calls share rows or keys among workgroups (the rules are host code): the shapes where the shared form was
measured faster by a tenth and more, and those where it was slower ((B, H, N, d, c_q, causal)); split counts of decode."""
import ctypes as C

import pytest

from flash_multi_token_attention_amd import _lib
from flash_multi_token_attention_amd.conv_attn import ops


def _bytes(fn, B, H, N, d, c_q, causal):
    c_k = {3: 3, 6: 11, 7: 7, 11: 11}[c_q]
    desc = _lib.Desc(B, H, N, N, d, c_q, c_k, 0.1, int(causal), _lib.BF16, _lib.BF16, 1, 0)
    return getattr(_lib.load(), fn)(C.byref(desc))


BWD = [
    # shared, unsplit in us
    ((2, 8, 1531, 64, 11, True), True), ((1, 8, 2048, 64, 7, True), True), ((1, 8, 640, 64, 6, True), True),     # 36 / 56
    ((1, 1, 8000, 128, 6, True), True), ((1, 4, 6000, 64, 6, True), True), ((1, 8, 6000, 64, 11, True), True),   # 612 / 704
    ((1, 8, 2048, 64, 6, False), True),                                                                          # 133 / 152
    ((1, 8, 8000, 128, 6, True), False), ((1, 12, 5000, 64, 6, True), False), ((1, 12, 5000, 128, 11, True), False),   # 842 / 712
    ((1, 8, 6000, 128, 3, True), False), ((4, 16, 1024, 64, 6, True), False), ((1, 4, 8192, 64, 6, True), False),
    ((5, 16, 1024, 64, 6, True), False), ((1, 8, 608, 64, 6, True), False),
]
FWD = [
    ((1, 8, 2048, 64, 7, True), True), ((1, 8, 1000, 128, 6, True), True), ((1, 1, 8000, 64, 6, True), True),     # 53 / 157
    ((1, 4, 8000, 64, 6, True), True), ((1, 6, 6000, 64, 6, True), True), ((1, 2, 8000, 128, 6, False), True),    # 149 / 196
    ((2, 16, 2048, 64, 6, True), False), ((2, 16, 2048, 128, 3, True), False), ((1, 8, 8000, 128, 6, True), False),   # 277 / 246
    ((1, 16, 1000, 64, 3, True), False), ((1, 24, 1600, 64, 11, True), False), ((1, 3, 8000, 128, 6, False), False),   # 215 / 196
    ((1, 1, 8192, 64, 6, True), False), ((5, 16, 1024, 64, 6, True), False), ((1, 8, 900, 64, 6, True), False),
]


@pytest.mark.parametrize("shape,shared", BWD)
def test_backward(shape, shared):
    assert (_bytes("convattn_bwd_split_workspace_bytes", *shape) > 0) == shared


@pytest.mark.parametrize("shape,shared", FWD)
def test_forward(shape, shared):
    assert (_bytes("convattn_fwd_split_workspace_bytes", *shape) > 0) == shared


@pytest.mark.parametrize("args,low,high", [
    # B, H, Nk, ragged, d: measured within 5 % of the best count between low and high
    ((1, 8, 65536, False, 128), 32, 32), ((32, 32, 8192, False, 128), 1, 1), ((32, 32, 8192, False, 64), 2, 8),
    ((16, 8, 40000, False, 32), 4, 4), ((32, 8, 20000, False, 32), 2, 2), ((32, 8, 65000, True, 64), 8, 48),
    ((24, 32, 8192, True, 64), 2, 6), ((4, 8, 700, False, 64), 2, 2), ((64, 32, 300, False, 64), 1, 1),
])
def test_decode_split_counts(args, low, high):
    B, H, Nk, ragged, d = args
    assert low <= ops.default_k_splits(B, H, Nk, ragged, d) <= high
    # one sequence has no others that could be shorter
    assert ops.default_k_splits(1, H, Nk, True, d) == ops.default_k_splits(1, H, Nk, False, d)


@pytest.mark.parametrize("Nk", [1, 128, 129, 513, 2048, 40000])
@pytest.mark.parametrize("asked", [1, 2, 16, 32, 700])
def test_an_explicit_count_does_not_follow_the_batch(Nk, asked):
    lib = _lib.load()
    counts = {lib.convattn_decode_step_splits(B, H, Nk, d, asked) for B, H in ((1, 1), (2, 2), (8, 32), (64, 64)) for d in (32, 64, 128)}
    assert counts == {min(asked, -(-Nk // 128))}
