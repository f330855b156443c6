"""GPU parity: document-masked GQA attention forward and backward vs the oracle.

Tolerance: outputs and gradients within 2e-2 absolute (plus 2e-2 relative for
entries above 1, where bf16 storage itself rounds by more than 2e-2), bf16
operands with fp32 accumulation, against the float64 oracle on the same
bf16 inputs.  Padding rows (doc_id -1) follow FlexAttention's mask_mod
semantics (a pad attends to earlier pads); the eager convention (pad rows 0)
is checked separately on real rows.
"""

from __future__ import annotations

import math

import numpy as np
import pytest
import torch

from oracle import attention as OA
from packbalance_amd.data import workloads as W
from packbalance_amd.model.attention import (
    attention_forward,
    build_doc_block_mask,
    doc_attention,
    flex_attention,
)

pytestmark = pytest.mark.gpu
TOL = 2e-2


def _close(got, want, what):
    torch.testing.assert_close(got.detach().float().cpu(), want.float(), atol=TOL, rtol=TOL,
                               msg=lambda m: f"{what}: {m}")


def _inputs(B, Hq, Hkv, S, D, dev, *, seed=0, model_layout=True):
    """q/k/v as the model makes them: .transpose(1, 2) views of [B, S, H, D] memory."""
    g = torch.Generator().manual_seed(seed)
    if model_layout:
        q = torch.randn(B, S, Hq, D, generator=g).to(dev, torch.bfloat16).transpose(1, 2)
        k = torch.randn(B, S, Hkv, D, generator=g).to(dev, torch.bfloat16).transpose(1, 2)
        v = torch.randn(B, S, Hkv, D, generator=g).to(dev, torch.bfloat16).transpose(1, 2)
        do = torch.randn(B, S, Hq, D, generator=g).to(dev, torch.bfloat16).transpose(1, 2)
    else:
        q = torch.randn(B, Hq, S, D, generator=g).to(dev, torch.bfloat16)
        k = torch.randn(B, Hkv, S, D, generator=g).to(dev, torch.bfloat16)
        v = torch.randn(B, Hkv, S, D, generator=g).to(dev, torch.bfloat16)
        do = torch.randn(B, Hq, S, D, generator=g).to(dev, torch.bfloat16)
    return q, k, v, do


def _run(q, k, v, do, doc, **kw):
    qr, kr, vr = (t.detach().requires_grad_(True) for t in (q, k, v))
    out = doc_attention(qr, kr, vr, doc, **kw)
    out.backward(do)
    return out, qr.grad, kr.grad, vr.grad


def _check(q, k, v, do, doc, what, **kw):
    out, dq, dk, dv = _run(q, k, v, do, doc, **kw)
    ref = OA.attention(q, k, v, doc.cpu(), do)
    _close(out, ref["out"], f"{what} out")
    _close(dq, ref["dq"], f"{what} dq")
    _close(dk, ref["dk"], f"{what} dk")
    _close(dv, ref["dv"], f"{what} dv")


def test_reference_flex_test_case(dev) -> None:
    """tests/test_attention.py:58-73 of the reference: fp32 q/k/v [1,2,64,16]."""
    torch.manual_seed(0)
    q = torch.randn(1, 2, 64, 16, device=dev)
    k = torch.randn(1, 2, 64, 16, device=dev)
    v = torch.randn(1, 2, 64, 16, device=dev)
    doc_ids = torch.tensor([[0] * 20 + [1] * 44], device=dev)
    mask = build_doc_block_mask(doc_ids, n_heads=2)
    out = flex_attention(q, k, v, block_mask=mask)
    assert out.dtype == torch.float32 and out.shape == q.shape
    ref = OA.attention(q, k, v, doc_ids.cpu(), semantics="eager")["out"]
    # fp32 inputs run the fp32 kernels (the reference computes fp32 tensors in fp32)
    torch.testing.assert_close(out.cpu().double(), ref, atol=2e-5, rtol=2e-4)


@pytest.mark.parametrize(
    "B,Hq,Hkv,S,D,docs",
    [
        (1, 2, 2, 64, 16, [20, 44]),
        (1, 4, 2, 256, 32, [60, 50, 100, 46]),  # cfg1 shape
        (2, 4, 1, 300, 64, [100, 150, -50]),  # -n: n pad tokens (doc -1)
        (1, 12, 4, 2048, 64, "cfg2"),  # cfg2 shape, heavy-tail pack
        (1, 8, 8, 1000, 128, [1000]),  # one dense doc, S not a tile multiple
        (1, 6, 2, 200, 128, [1] * 50 + [150]),  # single-token documents
        (3, 4, 4, 130, 100, [64, 66]),  # head dim not a multiple of 16
        (1, 4, 2, 130, 100, [64, 66]),  # split dK/dV, element-wise reduce (D % 8 != 0)
        (1, 8, 2, 1024, 128, [300, 1, 400, -323]),  # pipelined path, 32 query rows per wave
        (2, 16, 4, 2048, 64, "cfg2"),  # 32 x 32 tiles, lists shared by two and four waves
        (1, 12, 4, 2048, 64, [2048]),  # one dense document: lists of up to 64 tiles
        (2, 6, 2, 1536, 64, [1000, 536]),
        # head-split dK/dV with KV lists of >= 16 steps (kKvChunkSteps) walked
        # as two halves:
        (1, 8, 2, 2048, 128, [1100, -948]),  # a long document then padding
        # the threshold itself: the 512-token document's first KV tile has a
        # 16-step list (two halves), every other tile 14 steps or fewer (whole)
        (1, 8, 2, 1024, 64, [512, 448, -64]),
        (1, 8, 2, 1024, 128, [512, 448, -64]),
        # lengths that end in every part of a 64-row tile, head dims padded to 64 and 128
        (1, 4, 2, 1, 64, [1]),
        (2, 4, 2, 65, 64, [40, 25]),
        (2, 3, 1, 95, 128, [90, -5]),
        (1, 4, 4, 97, 96, [33, 64]),
        (2, 6, 2, 191, 40, [100, 91]),
        (1, 12, 4, 1999, 64, [1200, 300, 499]),  # shared lists of a ragged length
    ],
)
def test_attention_matches_oracle(B, Hq, Hkv, S, D, docs, dev) -> None:
    if docs == "cfg2":
        packs = W.cfg2_steps(1)[0][:B]
    else:
        pad = sum(-d for d in docs if d < 0)
        packs = [[d for d in docs if d > 0]] * B
        assert sum(packs[0]) + pad == S
    doc = W.doc_ids_from_lengths(packs, S).to(dev)
    q, k, v, do = _inputs(B, Hq, Hkv, S, D, dev, seed=S + D)
    _check(q, k, v, do, doc, f"B{B} Hq{Hq} Hkv{Hkv} S{S} D{D}")


def test_attention_contiguous_layout_and_scale(dev) -> None:
    """Contiguous [B, H, S, D] views and a non-default scale (0.3 = 2.4x 1/sqrt(64)).

    The gradients grow with the scale (dQ, dK carry it as a factor and P gets
    sharper), and their error is dominated by the bf16 rounding of O entering
    D = rowsum(dO * O) -- present in any bf16-output implementation -- so the
    absolute gradient tolerance is scaled by scale * sqrt(D) = 2.4 here.
    """
    q, k, v, do = _inputs(1, 4, 2, 192, 64, dev, model_layout=False)
    doc = W.doc_ids_from_lengths([[70, 122]], 192).to(dev)
    out, dq, dk, dv = _run(q, k, v, do, doc, scale=0.3)
    ref = OA.attention(q, k, v, doc.cpu(), do, scale=0.3)
    _close(out, ref["out"], "out")
    # The north star's 2e-2 bar, against the oracle whose delta is formed
    # from the stored bf16 output (as the reference's own backward forms it).
    stored = OA.attention(q, k, v, doc.cpu(), do, scale=0.3, delta_out=out.detach().cpu())
    for got, name in ((dq, "dq"), (dk, "dk"), (dv, "dv")):
        _close(got, stored[name], f"{name} (delta from the stored output)")
    gtol = TOL * 0.3 * math.sqrt(64)
    for got, name in ((dq, "dq"), (dk, "dk"), (dv, "dv")):
        torch.testing.assert_close(got.detach().float().cpu(), ref[name].float(), atol=gtol,
                                   rtol=TOL, msg=lambda m, n=name: f"{n}: {m}")


def test_attention_noncontiguous_documents(dev) -> None:
    """A document id may appear in several runs: the mask compares ids, not ranges."""
    S = 160
    ids = torch.tensor([i % 3 for i in range(S)], device=dev)[None]
    q, k, v, do = _inputs(1, 2, 1, S, 32, dev, seed=7)
    _check(q, k, v, do, ids, "alternating docs")


def test_attention_noncontiguous_documents_pipelined(dev) -> None:
    """Same, at a shape the DMA-pipelined forward takes (S % 64 == 0, D 64)."""
    S = 256
    ids = torch.tensor([(i // 7) % 3 for i in range(S)], device=dev)[None]
    q, k, v, do = _inputs(1, 4, 2, S, 64, dev, seed=9)
    _check(q, k, v, do, ids, "alternating docs, pipelined")


def test_attention_forward_dispatch_and_eager_rows(dev) -> None:
    packs = [[90, 100]]
    S = 200  # 10 pad tokens
    doc = W.doc_ids_from_lengths(packs, S).to(dev)
    q, k, v, _ = _inputs(1, 4, 2, S, 64, dev, seed=3)
    bm = build_doc_block_mask(doc, 4)
    out = attention_forward(q, k, v, doc, block_mask=bm)
    eager = OA.attention(q, k, v, doc.cpu(), semantics="eager")["out"]
    real = doc[0].cpu() >= 0
    _close(out[:, :, real], eager[:, :, real], "real rows vs eager semantics")
    with pytest.raises(ValueError):
        attention_forward(q, k, v, doc, backend="nope")
    with pytest.raises(RuntimeError):
        attention_forward(q.cpu(), k.cpu(), v.cpu(), doc.cpu())
    with pytest.raises(RuntimeError, match="eager_attention"):
        attention_forward(q, k, v, doc, backend="eager")


def test_attention_deterministic(dev) -> None:
    doc = W.doc_ids_from_lengths([[300, 212]], 512).to(dev)
    q, k, v, do = _inputs(1, 8, 2, 512, 128, dev, seed=11)
    a = _run(q, k, v, do, doc)
    b = _run(q, k, v, do, doc)
    for x, y in zip(a, b):
        assert torch.equal(x, y)


@pytest.mark.parametrize(
    "B,Hq,Hkv,S,D",
    [
        (9, 32, 8, 1025, 128),  # paired dK/dV with kept dS, one row into a tile
        (9, 32, 8, 1087, 96),  # the same, head dim padded, one row short of a tile
        (10, 16, 8, 1056, 128),  # paired dK/dV without kept dS, a sub-tile wholly past the end
        (9, 12, 12, 639, 72),
        (12, 24, 8, 1000, 64),  # head dim 64: 128-row query tiles, the backward on 32 x 32
        (3, 12, 4, 2047, 56),  # 32 x 32 tiles in both
        (1, 9, 3, 1350, 64),
        (1, 4, 1, 801, 120),
    ],
)
def test_ragged_matches_padded(B, Hq, Hkv, S, D, dev) -> None:
    """The kernels with bounds (any length, head dims that are multiples of 8) against
    the unbounded ones on the same values: the length padded to a multiple of 64 with
    another document, the head dim padded with zeros.  Both sides round fp32 sums that
    differ in order only, so the relative 2-norm stays within one bf16 rounding on
    either side (2 x 2^-9)."""
    Sp, Dp = -(-S // 64) * 64, 64 if D <= 64 else 128
    g = torch.Generator(device=dev).manual_seed(S * D)

    def heads(h):  # [B, S, H, D] memory; columns past D are zero
        t = torch.randn(B, Sp, h, Dp, device=dev, generator=g).to(torch.bfloat16)
        t[..., D:] = 0
        return t.transpose(1, 2)

    q, k, v, do = heads(Hq), heads(Hkv), heads(Hkv), heads(Hq)
    packs = [W.fill_sequential(np.random.default_rng(S + b), S, np.log(300), 1.0, 1, S)
             for b in range(B)]
    doc = W.doc_ids_from_lengths(packs, S).to(dev)
    doc_p = torch.full((B, Sp), 1 << 40, dtype=torch.int64, device=dev)
    doc_p[:, :S] = doc
    do_p = do.clone()
    do_p[:, :, S:] = 0
    want = _run(q, k, v, do_p, doc_p, scale=D ** -0.5)
    cut = [t.transpose(1, 2)[:, :S, :, :D].contiguous().transpose(1, 2) for t in (q, k, v, do)]
    for layout in ("dense", "view"):
        if layout == "view":  # rows of the padded memory
            cut = [t[:, :, :S, :D] for t in (q, k, v, do)]
        got = _run(*cut, doc, scale=D ** -0.5)
        for name, a, b in zip(("out", "dq", "dk", "dv"), got, want):
            b = b[:, :, :S, :D].double()
            err = (a.double() - b).norm() / b.norm()
            assert err <= 2 ** -8, f"{layout} {name}: {err:.2e}"


@pytest.mark.parametrize(
    "B,Hq,Hkv,S,D",
    [
        (9, 32, 8, 1025, 128),  # a full grid of a length that is no multiple of 64
        (9, 32, 8, 1024, 96),  # of a padded head dim
    ],
)
def test_ds_from_fp32_p_on_full_grids(B, Hq, Hkv, S, D, dev) -> None:
    """Outside whole 64-row tiles of head dim 128 the backward forms dS from the fp32 P.
    Rounding a normal value to bf16 leaves 1.66e-3 of its 2-norm (2^-8 / sqrt(3) of the
    mantissa's scale), so dq and dk, which see the rounding of dS, their own and a little
    of O's through delta, are sqrt(2) of that and some: 2.5e-3.  P rounded first would
    make it sqrt(3) and as much again: over 2.9e-3.  The bound lies between, at 2^-8.5."""
    packs = [W.fill_sequential(np.random.default_rng(S + b), S, np.log(300), 1.0, 1, S)
             for b in range(B)]
    doc = W.doc_ids_from_lengths(packs, S).to(dev)
    q, k, v, do = _inputs(B, Hq, Hkv, S, D, dev, seed=S)
    _, dq, dk, _ = _run(q, k, v, do, doc)
    b, g, G = 4, 3, Hq // Hkv
    sl, hs = slice(b, b + 1), slice(G * g, G * (g + 1))
    ref = OA.attention(q[sl, hs], k[sl, g : g + 1], v[sl, g : g + 1], doc[sl].cpu(), do[sl, hs])
    for name, got, want in (("dq", dq[sl, hs], ref["dq"]), ("dk", dk[sl, g : g + 1], ref["dk"])):
        err = float((got.cpu().double() - want).norm() / want.norm())
        assert err <= 2 ** -8.5, f"{name}: {err:.2e}"


@pytest.mark.parametrize(
    "B,Hq,Hkv,S,D",
    [
        (2, 12, 4, 1999, 64),  # 32 x 32 tiles, one wave a list share
        (1, 4, 2, 4100, 40),  # lists in chunks
        (12, 24, 8, 1000, 64),  # 128-row query tiles
        (1, 16, 4, 2047, 128),
    ],
)
@pytest.mark.parametrize("dense", [True, False])
def test_exact_max_of_peaked_scores(dense, B, Hq, Hkv, S, D, dev) -> None:
    """Scores of standard deviation 4: a row's output is mostly its largest P's.  Outside
    whole tiles of head dims 64 and 128 the running max is exact, so that P is 1 and its
    bf16 rounding exact; what is left is the output's own rounding (1.66e-3 of the 2-norm
    of normal values, 2^-8 / sqrt(3) of the mantissa's scale) and 0.5e-3 from the smaller
    P: 1.73e-3.  A P rounded against an older max adds its 1.66e-3 times the share of the
    largest one: 2.0e-3.  The bound lies between."""
    packs = [[S]] * B if dense else [
        W.fill_sequential(np.random.default_rng(S + b), S, np.log(200), 1.0, 1, S) for b in range(B)]
    doc = W.doc_ids_from_lengths(packs, S).to(dev)
    q, k, v, do = _inputs(B, Hq, Hkv, S, D, dev, seed=S)
    q = (q * 4).to(torch.bfloat16)
    with torch.no_grad():
        out = doc_attention(q, k, v, doc)
    G = Hq // Hkv
    ref = OA.attention(q[:1, G:2 * G], k[:1, 1:2], v[:1, 1:2], doc[:1].cpu(), do[:1, G:2 * G])["out"]
    err = float((out[:1, G:2 * G].cpu().double() - ref).norm() / ref.norm())
    assert err <= 1.85e-3, f"{err:.2e}"


@pytest.mark.parametrize(
    "B,Hq,Hkv,S,D,misaligned,kv_tile,split",
    [
        (1, 4, 2, 4160, 64, False, 64, True),  # whole tiles: lists in chunks, heads split
        (1, 4, 2, 4161, 64, False, 64, True),  # the same with bounds
        (1, 6, 2, 4200, 40, False, 64, True),
        (1, 4, 1, 4100, 24, False, 64, True),
        (1, 4, 1, 4100, 32, False, 64, True),  # (the forward register-staged)
        (1, 16, 1, 1024, 64, False, 64, True),  # one KV head of a short sequence
        (1, 16, 1, 1023, 48, False, 64, True),
        (1, 8, 8, 4160, 64, False, 64, False),  # two waves a KV tile, whole lists
        (1, 8, 8, 4133, 56, False, 64, False),
        (2, 8, 8, 4160, 64, False, 128, False),  # four
        (2, 8, 8, 4161, 64, False, 128, False),
        (1, 4, 2, 4161, 64, True, 64, True),  # rows without 16-byte alignment
        (1, 8, 8, 4133, 32, True, 64, False),
        (2, 8, 8, 4161, 48, True, 128, False),
    ],
)
def test_workgroup_kernels_to_head_dim_64(B, Hq, Hkv, S, D, misaligned, kv_tile, split, dev) -> None:
    """Head dims to 64 past the 32 x 32 tiles' grids, in every form that serves them: the
    tiles and the head split that pb_attn_config names, and all four results of one KV head
    against the oracle.  Outputs and gradients round bf16 values at most twice (P or dS, and
    the result; 1.66e-3 of the 2-norm each), dQ and dK see O's rounding through delta too:
    within 2^-8.5."""
    from packbalance_amd.model import attention as A

    c = A.attn_config(B, Hq, Hkv, S, D)
    assert c["tiles"][A.BWD_KV] == (64, kv_tile) and c["tiles"][A.BWD_Q][1] == 64
    assert c["split"] == split
    if S > 4096:
        assert c["tiles"][A.FWD][1] == 64 and c["fwd_chunk"] > 0
    packs = [W.fill_sequential(np.random.default_rng(S + b), S, np.log(700), 1.0, 1, S)
             for b in range(B)]
    doc = W.doc_ids_from_lengths(packs, S).to(dev)
    q, k, v, do = _inputs(B, Hq, Hkv, S, D, dev, seed=S + Hq)
    if misaligned:
        def odd(t):
            mem = torch.zeros(B, S, t.shape[1], D + 1, dtype=t.dtype, device=dev)
            mem[..., :D] = t.transpose(1, 2)
            return mem[..., :D].transpose(1, 2)

        q, k, v, do = odd(q), odd(k), odd(v), odd(do)
    got = _run(q, k, v, do, doc)
    b, g, G = B - 1, Hkv - 1, Hq // Hkv
    sl, hs, ks = slice(b, b + 1), slice(G * g, G * (g + 1)), slice(g, g + 1)
    ref = OA.attention(q[sl, hs], k[sl, ks], v[sl, ks], doc[sl].cpu(), do[sl, hs])
    for name, t in zip(("out", "dq", "dk", "dv"), got):
        want = ref[name]
        err = float((t[sl, hs if name in ("out", "dq") else ks].detach().cpu().double()
                     - want).norm() / want.norm())
        assert err <= 2 ** -8.5, f"{name}: {err:.2e}"


@pytest.mark.parametrize(
    "B,Hq,Hkv,S,D,mu,misaligned",
    [
        (1, 4, 2, 4096, 64, 1e9, False),  # few tiles: four waves a query tile, eight a KV tile
        (2, 4, 2, 4096, 64, 1e9, False),  # two, 64 steps a wave; four
        (1, 2, 1, 4096, 64, 40, False),  # few heads a group: the backward splits them instead
        (1, 9, 3, 2047, 56, 1e9, False),  # eight waves a KV tile, a ragged length
        (1, 16, 4, 3072, 64, 900, False),  # the most KV tiles of eight waves
        (2, 12, 4, 2048, 64, 200, False),  # dK/dV lists shared by four waves
        (4, 16, 16, 2017, 64, 500, False),  # by two
        (8, 16, 16, 2048, 48, 150, False),  # by none
        (9, 16, 16, 2048, 48, 150, False),  # past the backward's largest grid
        (1, 64, 8, 4096, 40, 700, False),  # G = 8, the longest walks of four waves
        (5, 8, 1, 777, 64, 90, False),  # G = 8, split by head in the backward
        (8, 12, 4, 2048, 64, 300, False),  # the largest forward grid of these kernels
        (9, 12, 4, 2048, 64, 300, False),  # past it: another forward, the same backward
        (2, 4, 2, 333, 64, 60, True),  # rows without 16-byte alignment: copied first
        (2, 4, 2, 333, 32, 60, True),
        (4, 12, 4, 1999, 40, 300, True),
        (1, 32, 2, 1024, 64, 300, True),  # register-staged in the backward
    ],
)
def test_small_grid_matches_padded_head_dim(B, Hq, Hkv, S, D, mu, misaligned, dev) -> None:
    """The 32 x 32 tile kernels of small grids (head dims to 64) against the workgroup
    kernels on the same values with the head dim padded to 128 by zeros.  Either side
    rounds P or dS and then the output to bf16, each at most 2^-9 of the value and
    2^-9 / sqrt(3) in the mean square, so the relative 2-norm of the difference stays
    below 2 x 2^-9."""
    g = torch.Generator(device=dev).manual_seed(S * D + B)

    def heads(h):
        t = torch.randn(B, S, h, 128, device=dev, generator=g).to(torch.bfloat16)
        t[..., D:] = 0
        return t.transpose(1, 2)

    wide = [heads(Hq), heads(Hkv), heads(Hkv), heads(Hq)]
    packs = [W.fill_sequential(np.random.default_rng(S + b), S, np.log(mu), 1.0, 1, S)
             for b in range(B)]
    doc = W.doc_ids_from_lengths(packs, S).to(dev)
    want = _run(*wide, doc, scale=D ** -0.5)

    def cut(t):
        if not misaligned:
            return t[..., :D].transpose(1, 2).contiguous().transpose(1, 2)
        mem = torch.zeros(B, S, t.shape[1], D + 1, dtype=t.dtype, device=dev)
        mem[..., :D] = t[..., :D].transpose(1, 2)
        return mem[..., :D].transpose(1, 2)

    got = _run(*(cut(t) for t in wide), doc, scale=D ** -0.5)
    for name, a, b in zip(("out", "dq", "dk", "dv"), got, want):
        b = b[..., :D].double()
        err = (a.double() - b).norm() / b.norm()
        assert err <= 2 ** -8, f"{name}: {err:.2e}"


# Rows so short that no list has a part for a second (fourth, eighth) wave: fewer waves a
# workgroup.  Query tiles of 1, 7, 8, 11 and 12 list entries on small and large grids, KV
# tiles of 1 to 24 steps.
@pytest.mark.parametrize("B,Hq,Hkv,S,D", [
    (1, 4, 4, 20, 64), (2, 4, 2, 224, 64), (2, 4, 2, 225, 40), (64, 4, 4, 352, 40),
    (64, 4, 4, 353, 64), (64, 12, 4, 128, 64), (32, 12, 4, 200, 64), (1, 12, 4, 200, 64),
    (32, 4, 4, 200, 48), (33, 16, 2, 65, 64)])
def test_short_rows_match_padded_head_dim(B, Hq, Hkv, S, D, dev) -> None:
    for mu in (1e9, 40):
        test_small_grid_matches_padded_head_dim(B, Hq, Hkv, S, D, mu, False, dev)


@pytest.mark.parametrize("pack", [1, 0])
def test_attention_cfg3_pack(pack, dev) -> None:
    """cfg3 shape (S=8192, Hq=32, Hkv=8, D=128): all 8 packs run, one pack x one
    KV group (4 query heads) is checked against the oracle in full (fp32 oracle
    arithmetic for speed; its formulas are pinned in float64 on the CPU)."""
    packs = W.cfg3_packs()
    S, Hq, Hkv, D = 8192, 32, 8, 128
    doc = W.doc_ids_from_lengths(packs, S).to(dev)
    q, k, v, do = _inputs(8, Hq, Hkv, S, D, dev, seed=3)
    out, dq, dk, dv = _run(q, k, v, do, doc)
    g = 5  # KV head 5 -> query heads 20..23
    hs = slice(4 * g, 4 * g + 4)
    sl = slice(pack, pack + 1)
    ref = OA.attention(q[sl, hs], k[sl, g : g + 1], v[sl, g : g + 1], doc[sl].cpu(),
                       do[sl, hs], dtype=torch.float32)
    _close(out[sl, hs], ref["out"], "out")
    _close(dq[sl, hs], ref["dq"], "dq")
    _close(dk[sl, g : g + 1], ref["dk"], "dk")
    _close(dv[sl, g : g + 1], ref["dv"], "dv")
    assert torch.isfinite(out.float()).all() and torch.isfinite(dq.float()).all()


def test_attention_cfg3_sampled_rows_all_packs(dev) -> None:
    """cfg3 shape, every pack and every query head (all 8 KV groups): out and dQ
    at 24 sampled query rows per pack -- each document's first and last row,
    the pack's last row and random ones -- against the float64 row oracle."""
    packs = W.cfg3_packs()
    S, Hq, Hkv, D = 8192, 32, 8, 128
    doc = W.doc_ids_from_lengths(packs, S).to(dev)
    q, k, v, do = _inputs(8, Hq, Hkv, S, D, dev, seed=4)
    out, dq, _, _ = _run(q, k, v, do, doc)
    g = torch.Generator().manual_seed(12)
    rows = []
    for lens in packs:
        starts = torch.tensor([0] + list(torch.tensor(lens).cumsum(0)[:-1]))
        ends = torch.tensor(lens).cumsum(0) - 1
        pick = torch.cat([starts[:4], ends[:4], torch.tensor([S - 1]),
                          torch.randint(0, S, (15,), generator=g)])
        rows.append(pick.unique())
    ref = OA.attention_rows(q, k, v, doc.cpu(), do, rows)
    for b in range(8):
        _close(out[b][:, rows[b]], ref["out"][b], f"pack {b} out")
        _close(dq[b][:, rows[b]], ref["dq"][b], f"pack {b} dq")


@pytest.mark.parametrize("layout", ["mixed", "noncontiguous"])
def test_attention_large_grid_layouts(layout, dev) -> None:
    """A large-grid D 128 shape (>= 2048 query tiles per launch, no KV split) with
    long and single-token documents and a padded tail, or document ids that
    recur in several runs; every head of one KV group is checked in full
    against the oracle."""
    S, Hq, Hkv, D = 8192, 32, 8, 128
    if layout == "mixed":
        doc = W.doc_ids_from_lengths([[3000, 1, 1, 700, 64, 1990, 33, 2000]], S)  # 403 pad
    else:
        doc = torch.tensor([[(i // 300) % 5 for i in range(S)]])
    doc = doc.to(dev)
    q, k, v, do = _inputs(1, Hq, Hkv, S, D, dev, seed=21)
    out, dq, dk, dv = _run(q, k, v, do, doc)
    g = 3
    hs = slice(4 * g, 4 * g + 4)
    ref = OA.attention(q[:, hs], k[:, g : g + 1], v[:, g : g + 1], doc.cpu(), do[:, hs],
                       dtype=torch.float32)
    _close(out[:, hs], ref["out"], "out")
    _close(dq[:, hs], ref["dq"], "dq")
    _close(dk[:, g : g + 1], ref["dk"], "dk")
    _close(dv[:, g : g + 1], ref["dv"], "dv")
    assert torch.isfinite(out.float()).all()


def test_attention_kept_ds_two_quads_per_kv_head(dev) -> None:
    """Kept-dS backward with G = 8 (each KV head's dS blocks hold two quads of
    query heads, and two dQ workgroups read them), lognormal packs and a
    padded tail: every query head of KV head 1, pack 2, against the oracle."""
    B, Hq, Hkv, S, D = 8, 16, 2, 4096, 128
    rng = np.random.default_rng(5)
    lens = [W.fill_sequential(rng, S, np.log(512), 1.0, 16, S) for _ in range(B)]
    lens[2] = lens[2][:-1]  # padded tail
    doc = W.doc_ids_from_lengths(lens, S).to(dev)
    q, k, v, do = _inputs(B, Hq, Hkv, S, D, dev, seed=8)
    out, dq, dk, dv = _run(q, k, v, do, doc)
    sl, g = slice(2, 3), 1
    hs = slice(8 * g, 8 * g + 8)
    ref = OA.attention(q[sl, hs], k[sl, g : g + 1], v[sl, g : g + 1], doc[sl].cpu(), do[sl, hs],
                       dtype=torch.float32)
    _close(out[sl, hs], ref["out"], "out")
    _close(dq[sl, hs], ref["dq"], "dq")
    _close(dk[sl, g : g + 1], ref["dk"], "dk")
    _close(dv[sl, g : g + 1], ref["dv"], "dv")
    assert torch.isfinite(dq.float()).all()


@pytest.mark.parametrize("S,D", [(1024, 64), (1024, 128), (4160, 64)])
@pytest.mark.parametrize("profile", ["rising", "falling"])
def test_attention_running_max_moves(profile, S, D, dev) -> None:
    """Scores that rise along the sequence (the forward's running max moves
    every few sub-tiles, by up to ~40 log2 units, taking the rescaling slow
    path) or fall (the first valid sub-tile holds the max, every later one
    takes the fast path), with documents that leave some lanes' first
    sub-tiles fully masked: on 32 x 32 tiles (head dim 64, short sequences) and on
    the pipelined kernels."""
    B, Hq, Hkv = 1, 4, 2
    g = torch.Generator().manual_seed(31 + D)
    pos = torch.arange(S, dtype=torch.float32) / S
    ramp = 6.0 * (pos if profile == "rising" else 1.0 - pos)
    q = 0.5 + 0.1 * torch.randn(B, S, Hq, D, generator=g)
    k = ramp[None, :, None, None] + 0.3 * torch.randn(B, S, Hkv, D, generator=g)
    v = torch.randn(B, S, Hkv, D, generator=g)
    do = torch.randn(B, S, Hq, D, generator=g)
    q, k, v, do = (t.to(dev, torch.bfloat16).transpose(1, 2) for t in (q, k, v, do))
    doc = W.doc_ids_from_lengths([[40, 300, 1, 400]], S).to(dev)  # then pad tokens
    out, dq, dk, dv = _run(q, k, v, do, doc)
    ref = OA.attention(q, k, v, doc.cpu(), do)
    what = f"{profile} scores, D {D}"
    _close(out, ref["out"], f"{what} out")
    _close(dk, ref["dk"], f"{what} dk")
    _close(dv, ref["dv"], f"{what} dv")
    # The north star's 2e-2 bar for dQ, against the oracle whose delta is
    # formed from the stored bf16 output (as the reference's own backward
    # forms it), so the bf16 rounding of O is on both sides.
    stored = OA.attention(q, k, v, doc.cpu(), do, delta_out=out.detach().cpu())
    _close(dq, stored["dq"], f"{what} dq (delta from the stored output)")
    # dQ = scale dS K grows with |K| (entries up to ~6 here, against ~1 in the
    # N(0, 1) cases), and so does its error, which the bf16 rounding of O in
    # rowsum(dO * O) dominates (present in any bf16-output implementation):
    # the absolute tolerance is scaled by the mean |K| entry (~3).
    torch.testing.assert_close(dq.detach().float().cpu(), ref["dq"].float(), atol=3 * TOL,
                               rtol=TOL, msg=lambda m: f"{what} dq: {m}")


def _bwd_abi(q, k, v, out, do, lse, doc, outs=None):
    """pb_attn_bwd through the C ABI on given forward results; dq / dk / dv as
    [B, S, H, D] memory seen as [B, H, S, D] (the model's layout)."""
    from packbalance_amd import _native as N
    from packbalance_amd.model import attention as A

    B, Hq, S, D = q.shape
    Hkv = k.shape[1]
    plans = A._plans(doc, Hq, Hkv, D, None)
    if outs is None:
        outs = (torch.empty(B, S, Hq, D, device=q.device, dtype=q.dtype).transpose(1, 2),
                torch.empty(B, S, Hkv, D, device=q.device, dtype=q.dtype).transpose(1, 2),
                torch.empty(B, S, Hkv, D, device=q.device, dtype=q.dtype).transpose(1, 2),
                torch.empty(max(1, plans["workspace"]), dtype=torch.uint8, device=q.device))
    dq, dk, dv, ws = outs
    pq, pk = plans[A.BWD_Q], plans[A.BWD_KV]
    N.call("pb_attn_bwd", N.BHSD.of(q), N.BHSD.of(k), N.BHSD.of(v), N.BHSD.of(out),
           N.BHSD.of(do), N.BHSD.of(dq), N.BHSD.of(dk), N.BHSD.of(dv), lse.data_ptr(),
           ws.data_ptr(), doc.data_ptr(), doc.stride(0), pq.counts.data_ptr(),
           pq.lists.data_ptr(), pk.counts.data_ptr(), pk.lists.data_ptr(), B, Hq, Hkv, S, D,
           1.0 / math.sqrt(D), N.PB_BF16, N.stream_ptr(q))
    return outs


def _fwd_abi(q, k, v, doc):
    from packbalance_amd import _native as N
    from packbalance_amd.model import attention as A

    B, Hq, S, D = q.shape
    Hkv = k.shape[1]
    plans = A._plans(doc, Hq, Hkv, D, None)
    out = torch.empty(B, S, Hq, D, device=q.device, dtype=q.dtype).transpose(1, 2)
    lse = torch.empty(B, Hq, S, device=q.device, dtype=torch.float32)
    fws = torch.empty(max(1, plans["fwd_workspace"]), dtype=torch.uint8, device=q.device)
    p = plans[A.FWD]
    N.call("pb_attn_fwd", N.BHSD.of(q), N.BHSD.of(k), N.BHSD.of(v), N.BHSD.of(out),
           lse.data_ptr(), fws.data_ptr(), doc.data_ptr(), doc.stride(0), p.counts.data_ptr(),
           p.lists.data_ptr(), B, Hq, Hkv, S, D, 1.0 / math.sqrt(D), N.PB_BF16,
           N.stream_ptr(q))
    return out, lse


def test_kept_ds_backward_packs_independent(dev) -> None:
    """The kept-dS backward (dK/dV storing dS, then dQ from it) is independent
    of the batch around a pack: the gradients of a 4-pack call equal, bit for
    bit, those of each pack alone, on the same forward results (per-pack
    offsets of the plans, the dS blocks, lse and delta)."""
    B, Hq, Hkv, S, D = 4, 32, 8, 8192, 128
    doc = W.doc_ids_from_lengths(W.cfg3_packs()[:B], S).to(dev)
    q, k, v, do = _inputs(B, Hq, Hkv, S, D, dev, seed=21)
    out, lse = _fwd_abi(q, k, v, doc)
    dq, dk, dv, _ = _bwd_abi(q, k, v, out, do, lse, doc)
    for b in range(B):
        sl = slice(b, b + 1)
        dq1, dk1, dv1, _ = _bwd_abi(q[sl], k[sl], v[sl], out[sl], do[sl], lse[sl],
                                    doc[sl].contiguous())
        for name, got, want in (("dq", dq[sl], dq1), ("dk", dk[sl], dk1), ("dv", dv[sl], dv1)):
            assert torch.equal(got, want), f"pack {b} {name} differs from the single-pack call"
    assert torch.isfinite(dq.float()).all() and torch.isfinite(dk.float()).all()


def test_kept_ds_backward_graph_replays(dev) -> None:
    """The kept-dS backward captured into a HIP graph: every replay, with eager
    work and synchronisations between them and the outputs poisoned before
    each, gives the eager call's gradients bit for bit."""
    B, Hq, Hkv, S, D = 2, 32, 8, 8192, 128
    doc = W.doc_ids_from_lengths(W.cfg3_packs()[1 : 1 + B], S).to(dev)
    q, k, v, do = _inputs(B, Hq, Hkv, S, D, dev, seed=22)
    out, lse = _fwd_abi(q, k, v, doc)
    want = [t.clone() for t in _bwd_abi(q, k, v, out, do, lse, doc)[:3]]
    torch.cuda.synchronize()
    outs = _bwd_abi(q, k, v, out, do, lse, doc)  # static outputs and workspace
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        _bwd_abi(q, k, v, out, do, lse, doc, outs)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        _bwd_abi(q, k, v, out, do, lse, doc, outs)
    for rep in range(3):
        for t in outs[:3]:
            t.fill_(float("nan"))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        for name, got, w in zip(("dq", "dk", "dv"), outs[:3], want):
            assert torch.equal(got, w), f"replay {rep}: {name} differs from the eager call"
        _ = (q.float() * 2).sum().item()  # eager work between replays


@pytest.mark.parametrize("D", [64, 128])
def test_empty_plan_rows(D, dev) -> None:
    """A caller's plan may leave a tile's list empty (pb_attn_plan never does): the rows of
    that query tile get zero outputs, lse -inf and zero dQ, the KV rows zero dK and dV, and
    the other tiles what they get with the full plan, on the 32 x 32 tiles of head dim 64 as
    on the workgroup kernels."""
    from packbalance_amd.model import attention as A

    B, Hq, Hkv, S = 1, 4, 4, 512
    doc = W.doc_ids_from_lengths([[300, 212]], S).to(dev)
    q, k, v, do = _inputs(B, Hq, Hkv, S, D, dev, seed=5)
    full, _ = _fwd_abi(q, k, v, doc)
    mask = A.DocPlans(doc)
    plans = A._plans(mask.doc_ids, Hq, Hkv, D, mask)
    qt, kt = A.attn_config(B, Hq, Hkv, S, D)["tiles"][A.FWD][0], plans[A.BWD_KV].kv_tile
    assert qt == plans[A.BWD_Q].q_tile and (qt == 32) == (D == 64)
    for p in {id(p): p for p in (plans[A.FWD], plans[A.BWD_Q])}.values():
        p.counts[0, 1] = 0
    plans[A.BWD_KV].counts[0, 2] = 0
    qr, kr, vr = (t.detach().requires_grad_(True) for t in (q, k, v))
    out = doc_attention(qr, kr, vr, mask.doc_ids, block_mask=mask)
    out.backward(do)
    rows = torch.zeros(S, dtype=torch.bool, device=dev)
    rows[qt:2 * qt] = True
    assert (out[:, :, rows] == 0).all() and torch.equal(out[:, :, ~rows], full[:, :, ~rows])
    assert torch.isfinite(out.float()).all()
    assert (kr.grad[:, :, 2 * kt:3 * kt] == 0).all() and (vr.grad[:, :, 2 * kt:3 * kt] == 0).all()
    assert (qr.grad[:, :, rows] == 0).all() and (qr.grad[:, :, ~rows] != 0).any()


@pytest.mark.parametrize("S,D", [(801, 128), (1472, 96), (4200, 40)])
def test_forward_without_workspace(S, D, dev) -> None:
    """Lengths and head dims of the bounded forward need no workspace: without one a list is
    not cut into chunks.  Either way rounds P and the output to bf16 once, so the two differ
    by at most two such roundings (2 x 2^-9 in the 2-norm)."""
    from packbalance_amd import _native as N
    from packbalance_amd.model import attention as A

    B, Hq, Hkv = 1, 4, 2
    doc = W.doc_ids_from_lengths([[S - 100, 100]], S).to(dev)
    q, k, v, _ = _inputs(B, Hq, Hkv, S, D, dev, seed=6)
    want, want_lse = _fwd_abi(q, k, v, doc)
    plans = A._plans(doc, Hq, Hkv, D, None)
    assert plans["fwd_workspace"] > 0 and A.attn_config(B, Hq, Hkv, S, D)["fwd_chunk"] > 0
    out, lse = torch.empty_like(want), torch.empty_like(want_lse)
    p = plans[A.FWD]
    N.call("pb_attn_fwd", N.BHSD.of(q), N.BHSD.of(k), N.BHSD.of(v), N.BHSD.of(out),
           lse.data_ptr(), None, doc.data_ptr(), doc.stride(0), p.counts.data_ptr(),
           p.lists.data_ptr(), B, Hq, Hkv, S, D, 1.0 / math.sqrt(D), N.PB_BF16, N.stream_ptr(q))
    assert (out.double() - want.double()).norm() <= 2 ** -8 * want.double().norm()
    torch.testing.assert_close(lse, want_lse, atol=1e-4, rtol=0)


@pytest.mark.parametrize("B,S,D", [(1, 33, 32), (2, 700, 64), (3, 257, 40)])
def test_misaligned_forward_without_workspace(B, S, D, dev) -> None:
    """32 x 32 tiles, rows without 16-byte alignment and no workspace to copy them to: the
    register-staged kernel reads them in place.  P and the output are rounded to bf16 once on
    either side (2 x 2^-9 in the 2-norm)."""
    from packbalance_amd import _native as N
    from packbalance_amd.model import attention as A

    Hq, Hkv = 4, 2
    doc = W.doc_ids_from_lengths([[S - 30, 30]] * B, S).to(dev)

    def odd(t):  # the same values one element past a 16-byte boundary
        b, h, s, d = t.shape
        buf = torch.empty(b * s * h * d + 8, dtype=t.dtype, device=dev)
        v = buf[1:1 + b * s * h * d].view(b, s, h, d).transpose(1, 2)
        return v.copy_(t)

    q, k, v, _ = _inputs(B, Hq, Hkv, S, D, dev, seed=8)
    want, want_lse = _fwd_abi(q, k, v, doc)
    cfg = A.attn_config(B, Hq, Hkv, S, D)
    assert cfg["fwd_workspace"] > 0 and cfg["tiles"][A.FWD] == (32, 32)
    q, k, v, out = odd(q), odd(k), odd(v), odd(torch.full_like(want, float("nan")))
    assert q.data_ptr() % 16 == 2
    lse = torch.empty_like(want_lse)
    p = A._plans(doc, Hq, Hkv, D, None)[A.FWD]
    N.call("pb_attn_fwd", N.BHSD.of(q), N.BHSD.of(k), N.BHSD.of(v), N.BHSD.of(out),
           lse.data_ptr(), None, doc.data_ptr(), doc.stride(0), p.counts.data_ptr(),
           p.lists.data_ptr(), B, Hq, Hkv, S, D, 1.0 / math.sqrt(D), N.PB_BF16, N.stream_ptr(q))
    assert (out.double() - want.double()).norm() <= 2 ** -8 * want.double().norm()
    torch.testing.assert_close(lse, want_lse, atol=1e-4, rtol=0)
