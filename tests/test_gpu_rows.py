"""The batched step's matrix kernels (2 to 16 rows over bf16 planes): the tokens
and the K/V rows of a batched decode against each sequence decoded alone.  Both
paths sum in f32 over exact products, about 1e-6 apart after three layers
(2-norm); the bound is 2e-5.  That does not see the third plane (dropping it
moves sums by about 1e-6 too): test_all_bits_of_every_operand does."""
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


def _one_hot(rows, cols, at, scale=1.0):
    """A matrix that copies column at[r] to row r, exactly: code 1 times a power of two."""
    codes = np.zeros((rows, cols), np.int8)
    if at is not None:
        codes[np.arange(rows), at] = 1
    return Q8, np.full(rows, scale, np.float32), codes.view(np.uint8), cols


def _bf16(x):
    return synth.bf16_round(x)


def _apart(a, b):
    """Relative 2-norm distance up to a common factor (the norms' 1/rms)."""
    a, b = np.asarray(a, np.float64), np.asarray(b, np.float64)
    return np.linalg.norm(a / np.linalg.norm(a) - b / np.linalg.norm(b))


@pytest.mark.parametrize("nseq", [2, 5, 6, 9, 16])  # (row, plane) columns; planes; 8 rows a workgroup and the rest
def test_all_bits_of_every_operand(ctx, nseq):
    """One step through matrices that copy columns: V of layer 0 is the embedding
    row, V of layer 1 has gone through the attention merge, o_proj, gate/up and
    down, each handing its values on as planes.  A value is rounded one to four
    times on its way (about 3e-8 each, as a mean): the bound is 2e-7.  Without the
    third plane, or with another row's, it is 2e-6 off."""
    H, F, Q, KV = 512, 1280, 512, 256
    rng = np.random.default_rng(nseq)
    pick = lambda rows, cols: rng.permutation(np.resize(rng.permutation(cols), rows))
    v0, o, up, down, v1 = pick(KV, H), pick(H, Q), pick(F, H), pick(H, F), pick(KV, H)
    zero = {"q": _one_hot(Q, H, None), "k": _one_hot(KV, H, None), "o": _one_hot(H, Q, None),
            "gate": _one_hot(F, H, None), "up": _one_hot(F, H, None), "down": _one_hot(H, F, None),
            "ln1": np.ones(H, np.float32), "ln2": np.ones(H, np.float32)}
    embed = rng.standard_normal((64, H)).astype(np.float32)
    embed[:, 0] = 8.0  # every gate reads this column: one factor for all of a row
    w = {"layers": [{**zero, "v": _one_hot(KV, H, v0), "o": _one_hot(H, Q, o),
                     "gate": _one_hot(F, H, np.zeros(F, int)), "up": _one_hot(F, H, up),
                     "down": _one_hot(H, F, down, 2.0 ** 30)},  # what down adds to is rounded away
                    {**zero, "v": _one_hot(KV, H, v1)}],
         "lm_head": _one_hot(64, H, pick(64, H)), "final_norm": np.ones(H, np.float32), "embed": embed}
    m = lib.Model(ctx, DecoderConfig(hidden=H, inter=F, layers=2, heads=4, kv_heads=2, head_dim=128, vocab=64, eps=1e-5,
                                     rope_theta=500000.0))
    m.load_weights(w)
    seqs = [m.seq(8) for _ in range(nseq)]
    first = [3 * i + 1 for i in range(nseq)]
    lib.decode_batch(seqs, first, [0] * nseq, 2, eos=())
    for s, t in zip(seqs, first):
        x = embed[t]
        got0, got1 = s.read_kv(0)[1].reshape(-1), s.read_kv(1)[1].reshape(-1)
        assert got0.size == KV and got1.size == KV
        out = np.repeat(got0.reshape(2, 1, 128), 2, axis=1).reshape(-1)  # one cached row: both heads of a group give V
        h1 = x + out[o]
        want0, want1 = x[v0], h1[up[down[v1]]]
        for got, want in ((got0, want0), (got1, want1)):
            two = _bf16(want) + _bf16(want - _bf16(want))
            assert _apart(two, want) > 6e-7
            assert _apart(got, want) < 2e-7, (t, _apart(got, want))
