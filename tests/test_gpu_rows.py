"""The batched step's matrix kernels (2 to 16 rows over bf16 planes): the tokens
and the K/V rows of a batched decode against each sequence decoded alone.  Both
paths sum in f32 over exact products, about 1e-6 apart after three layers
(2-norm); the bound is 2e-5."""
import numpy as np
import pytest

from rapidocrvl_amd import lib, synth
from rapidocrvl_amd.config import DecoderConfig

pytestmark = pytest.mark.gpu

Q8, Q4, Q6 = 1000, 1001, 1002


def _cfg(hidden, inter, heads, kv_heads):
    return DecoderConfig(hidden=hidden, inter=inter, layers=3, heads=heads, kv_heads=kv_heads, head_dim=128, vocab=1024,
                         eps=1e-5, rope_theta=500000.0)


ERNIE = _cfg(1024, 3072, 16, 2)
# K of 4 and 12 stages of 128 columns: waves without a stage, and with two
RAGGED = _cfg(512, 1536, 4, 1)
# 4 and 10 stages; 1,280 rows of gate and up
SMALL = _cfg(512, 1280, 4, 2)
# 5 and 33 stages: columns in 128s, not in 256s, and past the streaming GEMV's 4,096
ODD = _cfg(640, 4224, 5, 1)


@pytest.mark.parametrize("cfg,qtype,nseq", [
    (RAGGED, Q8, 2), (RAGGED, Q6, 3), (RAGGED, Q8, 4),   # (row, plane) columns
    (SMALL, Q4, 5), (SMALL, Q6, 5),                      # their last row
    (SMALL, Q4, 6), (SMALL, Q8, 8), (SMALL, Q6, 9),      # plane by plane; 8 rows a workgroup and the rest
    # shapes the streaming GEMV does not take (down; the 4-bit head): small batches too
    (SMALL, Q4, 2), (SMALL, Q8, 2), (SMALL, Q8, 3), (SMALL, Q6, 4),
    (ODD, Q4, 3), (ODD, Q6, 5), (ODD, Q4, 10), (ODD, Q8, 16),
    (SMALL, Q8, 16), (ERNIE, Q4, 3), (ERNIE, Q4, 9), (ERNIE, Q6, 16), (ERNIE, Q8, 2),
])
def test_rows_match_single_decode(ctx, cfg, qtype, nseq):
    m = lib.Model(ctx, cfg)
    m.load_weights(synth.make_weights(cfg, qtype, seed=31))
    n_new = 6
    lens = [1 + (5 * i) % 13 for i in range(nseq)]  # 1..13: residual kept in place and not
    prompts = [synth.prompt_ids(n, seed=300 + i, high=cfg.vocab) for i, n in enumerate(lens)]

    def prefilled(ids):
        s = m.seq(len(ids) + n_new + 4)
        return s, int(s.generate(ids, 1, eos=(), use_prefill=True)[0])

    batch, firsts = zip(*[prefilled(ids) for ids in prompts])
    got = lib.decode_batch(list(batch), list(firsts), lens, n_new, eos=())
    for i, ids in enumerate(prompts):
        s, first = prefilled(ids)
        assert list(got[i]) == list(s.decode_greedy(first, lens[i], n_new, eos=())), i
        for li in range(cfg.layers):
            for a, b in zip(batch[i].read_kv(li), s.read_kv(li)):
                err = np.linalg.norm(a - b) / np.linalg.norm(b)
                assert err < 2e-5, (i, li, err)


@pytest.mark.parametrize("nseq", [7, 11])
def test_head_pass_over_the_last_three_rows(ctx, nseq):
    # 512 columns and 1,000 rows: the greedy head runs 4-vector passes, the last
    # one over three sequences and a padding row past them
    cfg = DecoderConfig(hidden=512, inter=1536, layers=1, heads=4, kv_heads=1, head_dim=128, vocab=1000, eps=1e-5,
                        rope_theta=500000.0)
    m = lib.Model(ctx, cfg)
    m.load_weights(synth.make_weights(cfg, Q8, seed=33))
    prompts = [synth.prompt_ids(3 + i, seed=500 + i, high=cfg.vocab) for i in range(nseq)]
    seqs, want = [], []
    for ids in prompts:
        s = m.seq(len(ids) + 12)
        first = int(s.generate(ids, 1, eos=(), use_prefill=True)[0])
        want.append(list(s.decode_greedy(first, len(ids), 8, eos=())))
        s.truncate(len(ids))
        seqs.append((s, first))
    got = lib.decode_batch([s for s, _ in seqs], [f for _, f in seqs], [len(ids) for ids in prompts], 8, eos=())
    assert [list(g) for g in got] == want


# matrices without tile images (520 columns): each sequence its own GEMVs
UNTILED = _cfg(520, 1040, 4, 1)


def _stream(m, ids, n_new):
    """A prefilled sequence, its first token, and its stream decoded alone."""
    s = m.seq(len(ids) + n_new + 4)
    first = int(s.generate(ids, 1, eos=(), use_prefill=True)[0])
    want = list(s.decode_greedy(first, len(ids), n_new, eos=()))
    s.truncate(len(ids))
    return s, first, want


@pytest.mark.parametrize("nseq", [2, 3, 4])
def test_batch_without_tile_images(ctx, nseq):
    m = lib.Model(ctx, UNTILED)
    m.load_weights(synth.make_weights(UNTILED, Q8, seed=35))
    prompts = [synth.prompt_ids(1 + 3 * i, seed=700 + i, high=UNTILED.vocab) for i in range(nseq)]
    seqs, firsts, want = zip(*[_stream(m, ids, 8) for ids in prompts])
    got = lib.decode_batch(list(seqs), list(firsts), [len(ids) for ids in prompts], 8, eos=())
    assert [list(g) for g in got] == list(want)


@pytest.mark.parametrize("qtype,vocab", [(Q4, 1024), (Q4, 1000), (Q8, 1000)])
def test_continuous_batch_drains(ctx, qtype, vocab):
    # 6 members, then 4, 2 and 1, on shapes the streaming GEMV does not take; heads
    # on the small GEMM, one pass per member, and 4-vector passes
    cfg = DecoderConfig(hidden=512, inter=1280, layers=2, heads=4, kv_heads=2, head_dim=128, vocab=vocab, eps=1e-5,
                        rope_theta=500000.0)
    m = lib.Model(ctx, cfg)
    m.load_weights(synth.make_weights(cfg, qtype, seed=34))
    budgets = [4, 4, 9, 9, 14, 20]
    prompts = [synth.prompt_ids(2 + 3 * i, seed=600 + i, high=vocab) for i in range(len(budgets))]
    seqs, firsts, want = zip(*[_stream(m, ids, n) for ids, n in zip(prompts, budgets)])
    b = lib.Batch(m)
    for s, f, ids, n in zip(seqs, firsts, prompts, budgets):
        b.join(s, f, len(ids), n, eos=())
    left = [6]
    while left[-1]:
        left.append(b.step(20))
    assert left == [6, 4, 2, 1, 0]
    for s, w in zip(seqs, want):
        assert list(b.leave(s)) == w
    b.close()
