"""The few-row MFMA GEMM (kern_rows.hip) at the edges of its tiles and of the
row range it serves, through fg_forward and fg_step, against the CPU oracle.

Rows 5..256 run on it (fewer on the GEMV, more on the LDS-tiled GEMM); its
tiles are 16x16, 16x32, 32x32, 32x64 and 64x64, picked by the row count, and 8
wavefronts split K (K = 128: four 32-deep steps, so half of them have none).
Bounds: split operands carry 16 bits of an activation, so a logit is within a
few 2^-16 of max|logit| (5e-5 asked); one fp16 term carries 11 (2e-3 asked).
"""
import numpy as np
import pytest

from autoresearch_amd import engine
from autoresearch_amd.weights import Dims, rope_tables, seeded_weights, uniform_ids
from oracle import oracle as O

pytestmark = pytest.mark.gpu

TINY = Dims(n_layer=2, d_model=128, n_head=2, n_kv_head=1, head_dim=64, vocab=512)
SMALL = Dims(n_layer=2, d_model=384, n_head=3, n_kv_head=3, head_dim=128, vocab=1024)
# d_model / 16 = 136 sums of squares per row: more than a block's threads take in one pass
WIDE = Dims(n_layer=1, d_model=2176, n_head=34, n_kv_head=2, head_dim=64, vocab=256)


def model(d, maxpos):
    w = seeded_weights(d, 11)
    c, s = (t.reshape(-1) for t in rope_tables(maxpos, d.head_dim))
    m = engine.Model(d, stacks=w)
    m.set_rope(c, s)
    return m, w, c, s


def rel(a, b):
    return float(np.abs(a - b).max() / np.abs(b).max())


@pytest.mark.parametrize("d,B,T", [
    (TINY, 1, 5), (TINY, 1, 16), (TINY, 1, 17), (TINY, 3, 21), (TINY, 1, 256), (TINY, 1, 257),
    (SMALL, 1, 15), (SMALL, 2, 32), (SMALL, 1, 65), (SMALL, 1, 128), (SMALL, 1, 129),
    (SMALL, 3, 85), (WIDE, 1, 9), (WIDE, 1, 40)])
def test_forward_rows(d, B, T):
    m, w, c, s = model(d, T)
    ids = uniform_ids(21 + T, B * T, d.vocab)
    ref = O.gpt_forward(ids, c, s, w, d, B, T)
    lg, _ = m.forward(ids, B, T)
    assert rel(lg, ref) <= 5e-5
    m.set_forward_f16(True)
    lg16, _ = m.forward(ids, B, T)
    assert rel(lg16, ref) <= (2e-3 if B * T > 128 else 5e-5)
    m.close()


@pytest.mark.parametrize("B", [5, 16, 17, 40, 70])
def test_step_rows(B):
    d, P = SMALL, 6
    m, w, c, s = model(d, P + 1)
    ids = uniform_ids(31 + B, B * (P + 1), d.vocab).reshape(B, P + 1)
    kv = m.kv(B, P + 1)
    kv.step_multi(ids[:, :P], want_logits=False)
    lg, nxt = kv.step(ids[:, P])
    ref = O.gpt_forward(ids.reshape(-1), c, s, w, d, B, P + 1).reshape(B, P + 1, -1)[:, P]
    assert rel(lg, ref) <= 5e-5
    assert np.array_equal(nxt, lg.argmax(axis=1))
    kv.close()
    m.close()


@pytest.mark.parametrize("d", [TINY, SMALL])
@pytest.mark.parametrize("B,pos,T", [
    (1, 0, 2), (1, 0, 16), (1, 0, 17), (2, 15, 2), (1, 16, 16), (1, 31, 33), (3, 32, 5),
    (1, 255, 2), (1, 256, 16), (1, 257, 47), (2, 300, 20)])
def test_chunk_attention_rows(d, B, pos, T):
    """Chunks attended from the cache rows (k_attn_rows) at the edges of its
    16-query blocks, 32-key tiles and 8-tile rounds. bf16 caches round K and V
    to 8 bits (2^-9 of each at most; asked 4e-3 of max|logit|)."""
    n = pos + T
    m, w, c, s = model(d, n)
    ids = uniform_ids(41 + n, B * n, d.vocab).reshape(B, n)
    ref = O.gpt_forward(ids.reshape(-1), c, s, w, d, B, n).reshape(B, n, -1)[:, pos:]
    for kv16, tol in ((False, 5e-5), (True, 4e-3)):
        kv = m.kv(B, n + 3, bf16=kv16)
        if pos:
            kv.step_multi(ids[:, :pos], want_logits=False)
        lg, nxt = kv.step_multi(ids[:, pos:])
        assert rel(lg, ref) <= tol
        assert np.array_equal(nxt, lg[:, -1].argmax(axis=1))
        kv.close()
    m.close()


@pytest.mark.parametrize("d,B,T,pos,kv16", [
    (TINY, 1, 2, 0, False), (TINY, 1, 40, 3, False), (SMALL, 2, 3, 0, False), (SMALL, 5, 9, 7, True),
    (SMALL, 17, 20, 0, False), (TINY, 3, 300, 0, False)])
def test_chunk_without_logits(d, B, T, pos, kv16):
    """A chunk whose logits nobody takes runs its last layer and lm_head for
    one row a sequence: the same cache bit for bit, and the id that the full
    pass's last row has as its maximum (within the passes' 5e-5)."""
    n = pos + T
    m, w, c, s = model(d, n + 1)
    ids = uniform_ids(51 + n, B * n, d.vocab).reshape(B, n)
    full, fast = m.kv(B, n + 1, bf16=kv16), m.kv(B, n + 1, bf16=kv16)
    for kv in (full, fast):
        if pos:
            kv.step_multi(ids[:, :pos])
    lg, _ = full.step_multi(ids[:, pos:])
    none, nxt = fast.step_multi(ids[:, pos:], want_logits=False)
    assert none is None and fast.len == full.len == n
    for a, b in zip(full.read(), fast.read()):
        assert np.array_equal(a, b)
    last = lg[:, -1]
    best = last.max(axis=1)
    assert np.all(best - last[np.arange(B), nxt] <= 1e-4 * np.abs(last).max())
    # and on from there
    a, _ = full.step(nxt)
    b, _ = fast.step(nxt)
    assert np.array_equal(a, b)
    full.close()
    fast.close()
    m.close()


@pytest.mark.parametrize("d,B,pos,T,kv16", [
    (TINY, 1, 1190, 40, False),    # grouped KV: 1200 keys at most
    (TINY, 1, 1200, 65, False),    # head_dim 64, two query blocks, split key ranges
    (TINY, 1, 2540, 40, True), (SMALL, 1, 2530, 47, True),
    (SMALL, 70, 33, 50, False), (SMALL, 70, 33, 50, True)])  # 840 workgroups
def test_chunk_attention_from_planes(d, B, pos, T, kv16):
    """Chunks past what the cache-row attention takes (attn_rows_fits): the
    cached positions split into planes, k_attn_mfma after them, with the logits
    and without (the last layer then skips the planes: the same cache, and the
    id of the full pass's last row). Bounds as for the cache-row attention."""
    n = pos + T
    m, w, c, s = model(d, n)
    ids = uniform_ids(81 + n, B * n, d.vocab).reshape(B, n)
    ref = O.gpt_forward(ids.reshape(-1), c, s, w, d, B, n).reshape(B, n, -1)[:, pos:]
    full, fast = m.kv(B, n, bf16=kv16), m.kv(B, n, bf16=kv16)
    for kv in (full, fast):
        for p in range(0, pos, 1000 if B == 1 else 25):
            kv.step_multi(ids[:, p:min(p + (1000 if B == 1 else 25), pos)], want_logits=False)
    held = m.bytes()[1]
    lg, nxt = full.step_multi(ids[:, pos:])
    if B == 1:  # (no more rows than before: what grew are the planes)
        assert m.bytes()[1] - held >= 8 * n * d.n_kv_head * d.head_dim
    else:
        assert B * d.n_head * ((T + 15) // 16) > 640
    assert rel(lg, ref) <= (4e-3 if kv16 else 5e-5)
    assert np.array_equal(nxt, lg[:, -1].argmax(axis=1))
    none, nx2 = fast.step_multi(ids[:, pos:], want_logits=False)
    assert none is None
    for a, b in zip(full.read(), fast.read()):
        assert np.array_equal(a, b)
    last = lg[:, -1]
    assert np.all(last.max(axis=1) - last[np.arange(B), nx2] <= 1e-4 * np.abs(last).max())
    full.close()
    fast.close()
    m.close()


@pytest.mark.parametrize("d,B,T", [(TINY, 1, 1300), (TINY, 3, 1201), (SMALL, 2, 1400)])
def test_forward_attention_from_planes(d, B, T):
    """Forwards past the cache-row attention in split operands (head_dim 64 and
    128), with and without the positive-score counts: the same logits bit for
    bit; the counts differ from the oracle's at most by the scores whose sign is
    within rounding (1e-4 of sum |q_d k_d|: 16 bits of each operand)."""
    m, w, c, s = model(d, T)
    ids = uniform_ids(91 + T, B * T, d.vocab)
    ref, cnt, amb = O.gpt_forward_pos(ids, c, s, w, d, B, T, rel_tol=1e-4)
    lg, _ = m.forward(ids, B, T)
    assert rel(lg, ref) <= 5e-5
    lgp, npos = m.forward_pos(ids, B, T)
    assert np.array_equal(lg, lgp)
    assert np.all(np.abs(npos.astype(np.int64) - cnt) <= amb)
    m.close()


WIDE1 = Dims(n_layer=1, d_model=768, n_head=6, n_kv_head=6, head_dim=128, vocab=256)
VOCAB = Dims(n_layer=1, d_model=128, n_head=1, n_kv_head=1, head_dim=128, vocab=8192)


@pytest.mark.parametrize("d,B,T", [
    (WIDE1, 1, 450),    # QKV on 64x64 tiles
    (WIDE1, 2, 901),    # QKV on 64x128 tiles, a ragged last one
    (WIDE1, 2, 1390),   # residual GEMMs on 128x128 tiles
    (VOCAB, 1, 600),    # lm_head on 128x256 tiles
    (VOCAB, 1, 1100),   # fp16 lm_head on 256x256 tiles
    (VOCAB, 2, 801)])   # both
def test_forward_tiles(d, B, T):
    """Passes past the few-row GEMM at the tiles their sizes pick, and the
    cross-entropy: from lm_head's epilogue or the stored logits, with and
    without the logits asked for (the same bits), against the oracle's (a
    logit's bound moves a cross-entropy by at most twice that)."""
    m, w, c, s = model(d, T)
    ids = uniform_ids(61 + T, B * (T + 1), d.vocab).reshape(B, T + 1)
    x, tg = np.ascontiguousarray(ids[:, :-1]).reshape(-1), np.ascontiguousarray(ids[:, 1:]).reshape(-1)
    ref = O.gpt_forward(x, c, s, w, d, B, T)
    ref_nll = O.nll(ref.reshape(-1, d.vocab), tg, d.vocab)
    top = float(np.abs(ref).max())
    for f16, tol in ((False, 5e-5), (True, 2e-3)):
        m.set_forward_f16(f16)
        lg, nll = m.forward(x, B, T, targets=tg)
        assert rel(lg, ref) <= tol
        assert np.abs(nll.reshape(-1) - ref_nll).max() <= 2 * tol * top
        alone = m.eval_bpb(ids, np.ones(d.vocab, np.int32), batch=B, want_nll=True)["nll"]
        assert np.array_equal(alone.reshape(-1), nll.reshape(-1))
    m.close()


@pytest.mark.parametrize("d,T", [(SMALL, 600), (VOCAB, 1500), (TINY, 40)])
def test_workspace_is_what_a_pass_uses(d, T):
    """A new handle's first pass allocates and clears its workspace: fp32 rows
    and logits, the operand planes, the row norms' partial sums (a 16th of
    d_model up to 256 rows, a 64th past them), lm_head's partials, and nothing
    a pass of these rows never touches; 16 parts, rounded up to 64 KiB each. (A
    chunk whose attention reads the cache rows has no other scratch.)"""
    m, w, c, s = model(d, T)
    kv = m.kv(1, T)
    base = m.bytes()[1]
    kv.step_multi(uniform_ids(71, T, d.vocab).reshape(1, T), want_logits=False)
    D, qd, V = d.d_model, d.n_head * d.head_dim, d.vocab
    rows, prow = T, (T + 15) // 16 * 16
    need = 4 * rows * (D + 2 * qd + 4 * D + V + 5) + 4 * rows * qd + 4 * prow * (D + qd + 4 * D)
    need += 4 * max(min(rows, 256) * D // 16, rows * D // 64) + 8 * rows * V // 64
    said = m.bytes()[1] - base
    assert need <= said <= need + 16 * 65536, (need, said)
    kv.close()
    m.close()
