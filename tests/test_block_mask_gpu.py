"""GPU parity: document block tables are bit-exact.

Checked against (a) the golden fixtures produced by torch's
create_block_mask, and (b) the numpy oracle on the benchmark workloads
(cfg1 / cfg2 / cfg3 packs), including B > 1 through ``doc_block_tables``.
"""

from __future__ import annotations

from pathlib import Path

import numpy as np
import pytest
import torch

from oracle import block_mask as OB
from packbalance_amd.data import workloads as W
from packbalance_amd.model.attention import build_doc_block_mask, doc_block_tables

pytestmark = pytest.mark.gpu

GOLDEN = Path(__file__).resolve().parent / "golden" / "block_masks.npz"


def _assert_tables(bm_tables: dict, want: dict, what: str) -> None:
    for name in OB.TABLE_NAMES:
        got = bm_tables[name]
        got = got.cpu().numpy() if isinstance(got, torch.Tensor) else got
        assert got.dtype == np.int32, f"{what}:{name} dtype {got.dtype}"
        np.testing.assert_array_equal(got, want[name], err_msg=f"{what}:{name}")


def test_block_tables_match_torch_golden(dev) -> None:
    z = np.load(GOLDEN)
    for name in z["layouts"]:
        name = str(name)
        doc = torch.from_numpy(z[f"{name}/doc_ids"]).to(dev)
        heads = int(z[f"{name}/heads"])
        bm = build_doc_block_mask(doc[None], heads)
        assert bm.BLOCK_SIZE == (int(z[f"{name}/block"]),) * 2, name
        assert bm.seq_lengths == (doc.numel(), doc.numel())
        _assert_tables({n: getattr(bm, n) for n in OB.TABLE_NAMES},
                       {n: z[f"{name}/{n}"] for n in OB.TABLE_NAMES}, name)


@pytest.mark.parametrize("cfg", ["cfg1", "cfg2", "cfg3"])
def test_block_tables_on_benchmark_packs(cfg, dev) -> None:
    if cfg == "cfg1":
        packs, s, heads = W.cfg1_packs(), 256, 4
    elif cfg == "cfg2":
        packs, s, heads = W.cfg2_steps(2)[1], 2048, 12
    else:
        packs, s, heads = W.cfg3_packs(), 8192, 32
    docs = W.doc_ids_from_lengths(packs, s)
    block = OB.doc_block_size(s)
    # Per pack through the reference entry point (B = 1).
    for b in range(len(packs)):
        bm = build_doc_block_mask(docs[b : b + 1].to(dev), heads)
        want = OB.tables_closed(docs[b].numpy(), heads, block)
        _assert_tables({n: getattr(bm, n) for n in OB.TABLE_NAMES}, want, f"{cfg}[{b}]")
    # All packs at once (B > 1 extension).
    t = doc_block_tables(docs.to(dev), heads, block)
    for b in range(len(packs)):
        want = OB.tables_closed(docs[b].numpy(), heads, block)
        _assert_tables({n: t[n][b : b + 1] for n in OB.TABLE_NAMES}, want, f"{cfg}[B={b}]")


@pytest.mark.parametrize("seed", range(4))
def test_block_tables_random_layouts(seed, dev) -> None:
    rng = np.random.default_rng(100 + seed)
    s = int(rng.integers(1, 3000))
    doc = np.sort(rng.integers(0, max(1, s // 50), s))
    if seed % 2:
        doc = rng.permutation(doc)
    if seed >= 2 and s > 8:
        doc[-int(rng.integers(1, 8)):] = -1
    bm = build_doc_block_mask(torch.from_numpy(doc).to(dev), 3)
    block = bm.BLOCK_SIZE[0]
    want = OB.tables_dense(doc, 3, block)
    _assert_tables({n: getattr(bm, n) for n in OB.TABLE_NAMES}, want, f"seed{seed}")


@pytest.mark.parametrize("kind", ["distinct", "permuted", "short"])
def test_block_tables_many_documents_a_block(kind, dev) -> None:
    """Blocks of more documents than are compared one by one."""
    s = 1300
    doc = np.arange(s) // (5 if kind == "short" else 1)
    if kind == "permuted":
        doc = np.random.default_rng(4).permutation(doc // 3)
    bm = build_doc_block_mask(torch.from_numpy(doc).to(dev), 2)
    want = OB.tables_dense(doc, 2, bm.BLOCK_SIZE[0])
    _assert_tables({n: getattr(bm, n) for n in OB.TABLE_NAMES}, want, kind)


def test_build_doc_block_mask_rejects_batch(dev) -> None:
    with pytest.raises(ValueError):
        build_doc_block_mask(torch.zeros(2, 64, dtype=torch.long, device=dev), 2)


@pytest.mark.parametrize("q_tile,kv_tile,by_kv", [(128, 64, 0), (64, 128, 1), (64, 64, 0), (64, 64, 1)])
def test_attention_plans_match_oracle(q_tile, kv_tile, by_kv, dev) -> None:
    """pb_attn_plan lists == the closed-form tile classes, ascending, each entry
    tile << 2 | kind: 1 FULL, 2 CAUSAL (a partial tile in which every in-range
    pair with kv <= q shares a document, checked densely per tile), 0 PARTIAL."""
    from packbalance_amd import _native as N

    packs = W.cfg3_packs()[:3] + [[5000, 3000, 192]]
    s = 8192
    doc = W.doc_ids_from_lengths(packs, s).to(dev)
    b = doc.shape[0]
    nq, nk = -(-s // q_tile), -(-s // kv_tile)
    rows, cols = (nk, nq) if by_kv else (nq, nk)
    counts = torch.empty((b, rows), dtype=torch.int32, device=dev)
    lists = torch.full((b, rows, cols), -7, dtype=torch.int32, device=dev)
    ws = torch.empty(b * nq * nk, dtype=torch.uint8, device=dev)
    N.call("pb_attn_plan", doc.data_ptr(), doc.stride(0), b, s, q_tile, kv_tile, by_kv,
           counts.data_ptr(), lists.data_ptr(), ws.data_ptr(), N.stream_ptr(doc))
    counts, lists = counts.cpu().numpy(), lists.cpu().numpy()

    def one_doc(d, qi, kj):  # every in-range pair with kv <= q shares a document
        qa = np.arange(qi * q_tile, min((qi + 1) * q_tile, s))
        ka = np.arange(kj * kv_tile, min((kj + 1) * kv_tile, s))
        causal = qa[:, None] >= ka[None, :]
        return bool(np.all((d[qa][:, None] == d[ka][None, :])[causal]))

    kinds = set()
    for i in range(b):
        d = doc[i].cpu().numpy()
        cls = OB.classify_closed(d, q_tile, kv_tile)
        for r in range(rows):
            want = []
            for c in range(cols):
                qi, kj = (c, r) if by_kv else (r, c)
                k = cls[qi, kj]
                if k == OB.FULL:
                    want.append((c << 2) | 1)
                elif k == OB.PARTIAL:
                    want.append((c << 2) | (2 if one_doc(d, qi, kj) else 0))
            kinds.update(w & 3 for w in want)
            assert counts[i, r] == len(want), (i, r)
            assert lists[i, r, : len(want)].tolist() == want, (i, r)
    assert kinds == {0, 1, 2}


@pytest.mark.parametrize("q_tile,kv_tile", [(32, 32), (128, 64), (64, 128), (1024, 32), (7, 5)])
@pytest.mark.parametrize("s,kind", [(1, "sorted"), (97, "sorted"), (1025, "sorted"), (700, "mixed"),
                                    (1999, "padded"), (1999, "distinct"), (900, "permuted"),
                                    (1500, "short"), (1100, "clash")])
def test_plan_rows_match_dense(q_tile, kv_tile, s, kind, dev) -> None:
    """Both orientations of a plan against the dense mask: ids that recur in any order,
    one id per token (in order and not, and ids that share the hash bits of the sieve over a
    tile's runs), tiles longer than a wave, and tiles cut by the sequence end."""
    from packbalance_amd import _native as N

    rng = np.random.default_rng(s + q_tile)
    d = np.sort(rng.integers(0, max(1, s // 60), s)).astype(np.int64)
    if kind == "mixed":
        d = rng.permutation(d)
    if kind == "padded":
        d[-40:] = -1
    if kind in ("distinct", "permuted", "clash"):
        d = np.arange(s, dtype=np.int64)
    if kind == "permuted":
        d = rng.permutation(d)
    if kind == "clash":  # times the inverse of the hash's multiplier: ids whose product is small
        inv = pow(0x9E3779B97F4A7C15, -1, 1 << 64)
        d = np.array([(int(x) * inv) % (1 << 64) for x in d], dtype=np.uint64).view(np.int64)
    if kind == "short":
        d = np.repeat(np.arange(s // 5 + 1, dtype=np.int64), 5)[:s]
    doc = torch.from_numpy(d)[None].to(dev)
    nq, nk = -(-s // q_tile), -(-s // kv_tile)
    pos = np.arange(s)
    causal, same = pos[:, None] >= pos[None], d[:, None] == d[None]
    want = np.zeros((nq, nk), dtype=np.int64) - 1  # -1: empty
    for i in range(nq):
        for j in range(nk):
            qs, ks = slice(i * q_tile, (i + 1) * q_tile), slice(j * kv_tile, (j + 1) * kv_tile)
            c, e = causal[qs, ks], same[qs, ks]
            if (c & e).any():
                full = c.shape == (q_tile, kv_tile) and (c & e).all()
                want[i, j] = 1 if full else 2 if e[c].all() else 0
    for by_kv in (0, 1):
        w = want.T if by_kv else want
        counts = torch.empty((1, w.shape[0]), dtype=torch.int32, device=dev)
        lists = torch.full((1,) + w.shape, -7, dtype=torch.int32, device=dev)
        ws = torch.empty(nq * nk, dtype=torch.uint8, device=dev)
        N.call("pb_attn_plan", doc.data_ptr(), doc.stride(0), 1, s, q_tile, kv_tile, by_kv,
               counts.data_ptr(), lists.data_ptr(), ws.data_ptr(), N.stream_ptr(doc))
        for r in range(w.shape[0]):
            row = [(c << 2) | int(k) for c, k in enumerate(w[r]) if k >= 0]
            assert lists[0, r, :int(counts[0, r])].tolist() == row, (by_kv, r)


def test_rows_of_more_tiles_than_fit_in_lds(dev) -> None:
    """Plan rows and block tables of more than 16384 tiles (classes in the workspace first),
    against the mask itself: tiles of 1024 x 1 tokens both ways, and 1-token blocks."""
    from packbalance_amd import _native as N

    s, own = 16500, 1024
    rng = np.random.default_rng(8)
    d = np.sort(rng.integers(0, s // 90, s)).astype(np.int64)
    d[-30:] = -1
    doc = torch.from_numpy(d)[None].to(dev)
    pos = torch.arange(s, device=dev)
    n = -(-s // own)
    for by_kv in (0, 1):
        # row r: the own tile's tokens against every token of the other axis
        nq, nk, qt, kt = (s, n, 1, own) if by_kv else (n, s, own, 1)
        counts = torch.empty((1, n), dtype=torch.int32, device=dev)
        lists = torch.full((1, n, s), -7, dtype=torch.int32, device=dev)
        ws = torch.empty(nq * nk, dtype=torch.uint8, device=dev)
        N.call("pb_attn_plan", doc.data_ptr(), doc.stride(0), 1, s, qt, kt, by_kv,
               counts.data_ptr(), lists.data_ptr(), ws.data_ptr(), N.stream_ptr(doc))
        for r in range(n):
            o = pos[r * own:(r + 1) * own]
            causal = (o[:, None] <= pos[None]) if by_kv else (o[:, None] >= pos[None])
            same = doc[0, o][:, None] == doc[0][None]
            full = (causal & same).all(0) & (len(o) == own)
            kind = torch.where(full, 1, torch.where((same | ~causal).all(0), 2, 0))
            cols = torch.nonzero((causal & same).any(0))[:, 0]
            want = ((cols << 2) | kind[cols]).to(torch.int32)
            assert int(counts[0, r]) == len(want), (by_kv, r)
            assert torch.equal(lists[0, r, :len(want)], want), (by_kv, r)
    s = 16385
    t = doc_block_tables(doc[:, :s].contiguous(), 1, 1)
    pos = pos[:s]
    for q_rows in (False, True):  # (a 1-token tile is full or empty, never partial)
        a = "q" if q_rows else "kv"
        assert not t[f"{a}_num_blocks"].any()
        for r in (0, 1, 4095, 9000, s - 31, s - 2, s - 1):
            on = (doc[0, :s] == doc[0, r]) & ((pos >= r) if q_rows else (pos <= r))
            want = torch.cat([pos[on], pos[~on]]).to(torch.int32)
            assert int(t[f"full_{a}_num_blocks"][0, 0, r]) == int(on.sum()), (a, r)
            assert torch.equal(t[f"full_{a}_indices"][0, 0, r], want), (a, r)
            assert torch.equal(t[f"{a}_indices"][0, 0, r], pos.to(torch.int32)), (a, r)
