"""Backward whose workgroups share the row tiles of a key block, forward whose workgroups share the keys of a row tile: against
the unsplit forms, from small problems that are split on, with ragged ends, all windows and head dimensions."""
import ctypes as C

import pytest
import torch

from flash_multi_token_attention_amd import _lib
from flash_multi_token_attention_amd.conv_attn import ops
from tests.util import rand_case, rel_max, scale_of

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("B,H,N,d,c_q,c_k,causal", [
    (1, 2, 641, 64, 3, 3, True), (1, 3, 705, 128, 6, 11, True), (2, 8, 1531, 64, 11, 11, True), (1, 8, 1000, 128, 8, 15, True),
    (1, 4, 700, 32, 6, 5, False), (1, 2, 2049, 128, 9, 11, False), (1, 8, 1157, 32, 11, 7, True), (1, 1, 4000, 64, 6, 11, True),
    # an instance per tap slot count: 7 and 8 up to d = 64, 7 at 128; 9 and 10 taps in 11 slots
    (2, 8, 1531, 64, 7, 7, True), (1, 8, 700, 64, 8, 15, True), (1, 2, 1000, 32, 7, 7, False), (1, 8, 1153, 32, 8, 9, True),
    (1, 2, 1100, 64, 8, 7, False), (1, 4, 1300, 64, 9, 5, True), (1, 4, 1300, 32, 10, 3, True), (1, 8, 2048, 128, 7, 7, True),
    (1, 4, 1001, 128, 7, 15, False),
])
@pytest.mark.parametrize("out_dtype", [torch.float32, torch.bfloat16])
def test_split_equals_unsplit(B, H, N, d, c_q, c_k, causal, out_dtype, monkeypatch):
    Q, K, V, dO, W = (t.to(DEV) for t in rand_case(B, H, N, N, d, c_q, c_k, torch.bfloat16, seed=N + d))
    sc, pq, pk = scale_of(d), c_q - 1, (c_k - 1) // 2
    O, M, L = ops.forward(Q, K, V, W, sc, pq, pk, causal, out_dtype=torch.bfloat16)
    D, LSE = ops.bwd_preprocess(O, dO, M, L)
    lib, desc = _lib.load(), ops._desc(Q, K, W, sc, causal, out_dtype)
    split, fused = lib.convattn_bwd_split_workspace_bytes(C.byref(desc)), lib.convattn_bwd_fused_workspace_bytes(C.byref(desc))
    assert split > fused > 0
    args = (Q, K, V, dO, D, LSE, W, sc, pq, pk, causal, out_dtype)
    got = ops.backward(*args)
    again = ops.backward(*args)
    monkeypatch.setenv("CONVATTN_MAX_WORKSPACE_BYTES", str(fused))   # no room for the partials: the unsplit form
    want = ops.backward(*args)
    assert all(torch.equal(a, b) for a, b in zip(got, again))
    assert torch.equal(got[0], want[0])   # dS is the same, block by block
    tol = 1e-5 if out_dtype == torch.float32 else 1e-2
    for a, b in zip(got[1:], want[1:]):
        assert rel_max(a.float(), b.float()) <= (tol if a.dtype == out_dtype else 1e-5)


@pytest.mark.parametrize("B,H,N,d,c_q,c_k,causal", [
    (1, 2, 1100, 64, 3, 3, True), (2, 8, 1531, 64, 11, 11, True), (1, 8, 1000, 128, 8, 15, True), (1, 4, 1217, 32, 6, 17, False),
    (1, 2, 2049, 128, 9, 11, False), (1, 8, 1157, 32, 11, 7, True), (1, 1, 4000, 64, 6, 11, True), (1, 3, 1600, 128, 6, 11, True),
    (1, 8, 1200, 64, 7, 7, True), (1, 4, 1217, 32, 7, 17, False), (1, 3, 1600, 128, 7, 7, True), (1, 6, 1203, 64, 8, 9, True),
    (1, 4, 1001, 128, 7, 15, False),
])
@pytest.mark.parametrize("out_dtype", [torch.float32, torch.bfloat16])
def test_split_forward_equals_unsplit(B, H, N, d, c_q, c_k, causal, out_dtype, monkeypatch):
    Q, K, V, _, W = (t.to(DEV) for t in rand_case(B, H, N, N, d, c_q, c_k, torch.bfloat16, seed=N + d))
    args = (Q, K, V, W, scale_of(d), c_q - 1, (c_k - 1) // 2, causal, out_dtype)
    assert _lib.load().convattn_fwd_split_workspace_bytes(C.byref(ops._desc(Q, K, W, args[4], causal, out_dtype))) > 0
    got, again = ops.forward(*args), ops.forward(*args)
    monkeypatch.setenv("CONVATTN_MAX_WORKSPACE_BYTES", "1024")   # no room for the parts: the unsplit form
    want = ops.forward(*args)
    assert all(torch.equal(a, b) for a, b in zip(got, again))
    # (probabilities are rounded to bf16 relative to the exponent base, and a part may have another base)
    assert float((got[0].float() - want[0].float()).norm() / want[0].float().norm()) <= 4e-3
    assert rel_max(got[1], want[1]) <= 1e-6
    assert rel_max(got[1] + torch.log(got[2]), want[1] + torch.log(want[2])) <= 1e-5
