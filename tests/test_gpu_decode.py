"""Batched RNNT greedy decoding on the GPU (pk_rnnt_greedy_step) against the
oracle (oracle/rnnt.py, pinned in test_oracle_rnnt.py).

Decisions are argmaxes, so an implementation with other rounding may break a
near-tie the other way.  The bar is per decision: the oracle replays the GPU's
decisions (tokens per frame, then blank) at the same rounding points, and every
decision's logit must be within 4 eps (|max logit| + rms(logits)) of the
oracle's maximum, eps = 2^-10 fp16, 2^-7 bf16, 2^-17 fp32; at most 2% of the
decisions may differ from the oracle's own argmax.  Predictor state after
reset_slot: |got - ref| <= 4 eps (|ref| + rms).  Streams are independent of the
batch they are decoded in (bit-exact), and slots outside a batch are untouched.
"""

import numpy as np
import pytest
import torch

from oracle import rnnt
from parakeet_amd.modules.decoder import GreedyDecoder, Joiner, Predictor

pytestmark = pytest.mark.gpu

EPS = {torch.float16: 2.0**-10, torch.bfloat16: 2.0**-7, torch.float32: 2.0**-17}


def _model(vocab, enc_dim, layers, dt, cuda, seed, blank_bias=1.5, out_scale=4.0):
    torch.manual_seed(seed)
    pred = Predictor(640, 640, layers, vocab)
    joint = Joiner(enc_dim, 640, 640, num_classes=vocab)
    with torch.no_grad():
        joint.joint_net[2].weight.mul_(out_scale)
        joint.joint_net[2].bias[vocab] += blank_bias
    pred = pred.to(dt).to(cuda).eval().requires_grad_(False)
    joint = joint.to(dt).to(cuda).eval().requires_grad_(False)
    P = rnnt.RnntParams(pred.state_dict(), joint.state_dict(), layers)
    return pred, joint, P


def _tol(dt):
    return lambda lg: 4 * EPS[dt] * (np.abs(lg).max() + np.sqrt((lg**2).mean()))


@pytest.mark.parametrize(
    "dt,layers,vocab,enc_dim,blank_bias,T,compact",  # the bias gives a mix of tokens and blanks
    [
        (torch.float16, 1, 1026, 512, 1.5, 3, 0),
        (torch.bfloat16, 2, 1024, 1024, 3.5, 3, 0),
        (torch.float32, 1, 1026, 512, 1.5, 3, 0),
        (torch.bfloat16, 2, 1024, 1024, 3.5, 14, 0),  # the large model's 14 frames a step (config.py:25-31)
        (torch.float16, 1, 1026, 512, 1.5, 3, 1),  # compact mode: lists of the updating streams
        (torch.float32, 2, 1026, 512, 3.0, 3, 1),
    ],
)
def test_greedy_decode_matches_oracle_replay(cuda, dt, layers, vocab, enc_dim, blank_bias, T, compact):
    pred, joint, P = _model(vocab, enc_dim, layers, dt, cuda, seed=layers + enc_dim, blank_bias=blank_bias)
    S, B = 20, 12
    dec = GreedyDecoder(pred, joint, blank_id=vocab, num_slots=S)
    dec.compact = compact
    rng = np.random.default_rng(7)
    slots = rng.permutation(S)[:B]
    dec.reset_slot(slots)
    oracles = [rnnt.StreamDecoder(P, vocab, dtype=dt) for _ in range(B)]
    n_dec = n_diff = n_tok = n_blankframes = 0
    for step in range(4):
        lengths = rng.integers(0, T + 1, B)
        if step == 0:
            lengths[:] = T
        enc = torch.randn(B, T, enc_dim, generator=torch.Generator().manual_seed(step)).to(dt).to(cuda)
        got = dec.decode(slots, enc, lengths, frame_tokens=True)
        for b in range(B):
            frames = enc[b, : lengths[b]].double().cpu().numpy()
            n, worst, differ = oracles[b].replay(frames, got[b], _tol(dt))
            n_dec += n
            n_diff += differ
            n_tok += sum(len(t) for t in got[b])
            n_blankframes += sum(len(t) < 5 for t in got[b])
    assert n_tok > 20 and n_blankframes > 5, (n_tok, n_blankframes)  # both tokens and blanks occurred
    assert n_diff <= 0.02 * n_dec, f"{n_diff} of {n_dec} decisions differ from the oracle's argmax"


def test_reset_slot_gives_the_start_state(cuda):
    dt = torch.float16
    pred, joint, P = _model(1026, 512, 2, dt, cuda, seed=3)
    dec = GreedyDecoder(pred, joint, blank_id=1026, num_slots=6)
    dec.reset_slot([4, 1])
    ref_out, ref_h, ref_c = rnnt.init_state(P, 1026, dt)
    for s in (4, 1):
        for got, ref in ((dec.h[s], ref_h), (dec.c[s], ref_c)):
            g = got.double().cpu().numpy()
            rms = np.sqrt((ref**2).mean())
            assert (np.abs(g - ref) <= 4 * EPS[dt] * (np.abs(ref) + rms)).all()
        pp = dec.pred_proj[s].double().cpu().numpy()
        ref_pp = rnnt.pred_proj(P, ref_out, dt)
        assert (np.abs(pp - ref_pp) <= 4 * EPS[dt] * (np.abs(ref_pp) + np.sqrt((ref_pp**2).mean()))).all()
    assert not dec.h[[0, 2, 3, 5]].any()  # other slots untouched


def test_streams_are_independent_of_the_batch(cuda):
    """A stream's tokens and state do not depend on its position in the batch or
    its slot (bit for bit; the batch size is kept so the enc GEMM is the same
    kernel); slots outside the batch do not move."""
    dt = torch.float16
    pred, joint, _ = _model(1026, 512, 1, dt, cuda, seed=5)
    a = GreedyDecoder(pred, joint, blank_id=1026, num_slots=8)
    b = GreedyDecoder(pred, joint, blank_id=1026, num_slots=8)
    a.reset_slot(range(8))
    b.reset_slot(range(8))
    sa = np.array([0, 2, 4, 6, 7])
    perm = np.array([3, 0, 4, 1, 2])
    sb = np.array([5, 1, 3, 7, 0])  # stream i of a lives on slot sb[i] in b, at batch position inv[i]
    inv = np.argsort(perm)
    g = torch.Generator().manual_seed(9)
    for step in range(3):
        enc = torch.randn(5, 2, 512, generator=g).to(dt).to(cuda)
        lengths = np.array([2, 1, 2, 0, 2])
        ta = a.decode(sa, enc, lengths)
        before = b.h[[2, 4, 6]].clone()
        tb = b.decode(sb[perm], enc[torch.from_numpy(perm).to(cuda)], lengths[perm])
        assert [tb[inv[i]] for i in range(5)] == ta
        for i in range(5):
            assert torch.equal(a.h[sa[i]], b.h[sb[i]]) and torch.equal(a.c[sa[i]], b.c[sb[i]])
            assert torch.equal(a.pred_proj[sa[i]], b.pred_proj[sb[i]])
        assert torch.equal(b.h[[2, 4, 6]], before)


@pytest.mark.parametrize("dt,layers,n", [(torch.float16, 1, 128), (torch.bfloat16, 2, 128), (torch.bfloat16, 2, 150)])
def test_wide_lstm_tiles_match_narrow(cuda, dt, layers, n):
    """n streams in one batch (128; 150, whose last 32-stream tile is partial) take
    the LSTM launches of 32 streams a workgroup at a frame's first symbol (their
    16-stream tiles would leave CUs with two workgroups); the same streams as two
    half batches take 16-stream workgroups throughout.  Tokens and state agree bit
    for bit.  The joint's encoder projection is the identity, so the enc GEMM
    gives the same bits whatever kernel each batch size picks."""
    pred, joint, _ = _model(1024, 640, layers, dt, cuda, seed=11, blank_bias=2.5)
    with torch.no_grad():
        joint.enc.weight.copy_(torch.eye(640, dtype=dt))
        joint.enc.bias.zero_()
    a = GreedyDecoder(pred, joint, blank_id=1024, num_slots=n)
    b = GreedyDecoder(pred, joint, blank_id=1024, num_slots=n)
    a.reset_slot(range(n))
    b.reset_slot(range(n))
    g = torch.Generator().manual_seed(13)
    h = n // 2
    n_tok = 0
    for step in range(3):
        enc = (0.5 * torch.randn(n, 4, 640, generator=g)).to(dt).to(cuda)
        lengths = np.array([4 - (i % 3 == 0) for i in range(n)])
        ta = a.decode(np.arange(n), enc, lengths)
        tb = list(b.decode(np.arange(h), enc[:h], lengths[:h])) + list(b.decode(np.arange(h, n), enc[h:], lengths[h:]))
        assert [list(x) for x in ta] == [list(x) for x in tb], f"step {step}"
        assert torch.equal(a.h, b.h) and torch.equal(a.c, b.c) and torch.equal(a.pred_proj, b.pred_proj)
        n_tok += sum(len(x) for x in ta)
    assert n_tok > 100, n_tok  # tokens were emitted, so the LSTM launches did work


@pytest.mark.parametrize("blank_bias,expect", [(-50.0, "cap"), (50.0, "none")])
def test_symbol_cap_and_all_blank(cuda, blank_bias, expect):
    """A blank that never wins: every frame stops at max_symbols tokens
    (model_runner.py:422); a blank that always wins: no tokens."""
    dt = torch.float16
    pred, joint, _ = _model(1026, 512, 1, dt, cuda, seed=6, blank_bias=blank_bias)
    dec = GreedyDecoder(pred, joint, blank_id=1026, num_slots=4, max_symbols=5)
    dec.reset_slot(range(4))
    enc = torch.randn(4, 3, 512, generator=torch.Generator().manual_seed(1)).to(dt).to(cuda)
    got = dec.decode(range(4), enc, [3, 2, 1, 0], frame_tokens=True)
    for b, L in enumerate([3, 2, 1, 0]):
        assert len(got[b]) == L
        for toks in got[b]:
            assert len(toks) == (5 if expect == "cap" else 0)
            assert all(0 <= k < 1026 for k in toks)


def test_graph_replay_matches_direct_launches(cuda):
    """The recorded decode step replayed over persistent buffers gives the same
    tokens and state as the direct launches, step after step, with other work in
    between (a graph of the enc GEMM and every launch of the step)."""
    dt = torch.float16
    pred, joint, _ = _model(1026, 512, 1, dt, cuda, seed=8)
    a = GreedyDecoder(pred, joint, blank_id=1026, num_slots=10)
    b = GreedyDecoder(pred, joint, blank_id=1026, num_slots=10)
    slots = np.array([7, 1, 4, 9, 2, 0])
    a.reset_slot(slots)
    b.reset_slot(slots)
    g = torch.Generator().manual_seed(4)
    for step in range(5):
        enc = torch.randn(6, 2, 512, generator=g).to(dt).to(cuda)
        lengths = np.array([2, 2, 1, 0, 2, 1]) if step % 2 else None
        ta = a.decode(slots, enc, lengths)
        tb = b.decode(slots, enc, lengths, graph=True)
        assert ta == tb, f"step {step}"
        assert torch.equal(a.h, b.h) and torch.equal(a.c, b.c) and torch.equal(a.pred_proj, b.pred_proj)
        torch.cuda.synchronize()


def test_graph_replay_after_refresh_weights(cuda):
    """A decode step recorded before new weights are loaded replays with the new
    weights once refresh_weights() ran (same shapes: the decoder's buffers are
    updated in place), matching direct launches of a decoder built on them."""
    dt = torch.float16
    pred, joint, _ = _model(1026, 512, 1, dt, cuda, seed=9)
    pred2, joint2, _ = _model(1026, 512, 1, dt, cuda, seed=10)
    a = GreedyDecoder(pred, joint, blank_id=1026, num_slots=8)
    slots = np.array([3, 0, 6, 1])
    a.reset_slot(slots)
    g = torch.Generator().manual_seed(5)
    enc = torch.randn(4, 2, 512, generator=g).to(dt).to(cuda)
    a.decode(slots, enc, graph=True)  # records the step with the first weights
    with torch.no_grad():
        pred.load_state_dict(pred2.state_dict())
        joint.load_state_dict(joint2.state_dict())
    a.refresh_weights()
    b = GreedyDecoder(pred2, joint2, blank_id=1026, num_slots=8)
    a.reset_slot(slots)
    b.reset_slot(slots)
    for step in range(3):
        enc = torch.randn(4, 2, 512, generator=g).to(dt).to(cuda)
        ta = a.decode(slots, enc, graph=True)
        tb = b.decode(slots, enc)
        assert ta == tb, f"step {step}"
        assert torch.equal(a.h, b.h) and torch.equal(a.c, b.c) and torch.equal(a.pred_proj, b.pred_proj)
    torch.cuda.synchronize()


def test_out_of_range_slot_is_skipped_by_the_kernels(cuda):
    """A slot id outside the state arrays (a caller error the host wrapper
    rejects) reaching the kernels through the C ABI: the kernels treat that
    stream as absent -- no tokens, zero frame counts, no state read or written
    -- and the batch's other streams decode exactly as they would next to a
    valid stream (same batch size, so the same enc GEMM)."""
    dt = torch.float16
    pred, joint, _ = _model(1026, 512, 1, dt, cuda, seed=11)
    a = GreedyDecoder(pred, joint, blank_id=1026, num_slots=4)
    b = GreedyDecoder(pred, joint, blank_id=1026, num_slots=4)
    a.reset_slot(range(4))
    b.reset_slot(range(4))
    a._check_slots = lambda slots: np.ascontiguousarray(np.asarray(slots, dtype=np.int32).reshape(-1))
    enc = torch.randn(3, 3, 512, generator=torch.Generator().manual_seed(2)).to(dt).to(cuda)
    before = (a.h.clone(), a.c.clone(), a.pred_proj.clone())
    got = a.decode([0, 4, 2], enc, frame_tokens=True)
    ref = b.decode([0, 1, 2], enc, frame_tokens=True)
    assert got[1] == [[], [], []]
    assert got[0] == ref[0] and got[2] == ref[2]
    for s in (0, 2):
        assert torch.equal(a.h[s], b.h[s]) and torch.equal(a.c[s], b.c[s]) and torch.equal(a.pred_proj[s], b.pred_proj[s])
    for s in (1, 3):
        assert torch.equal(a.h[s], before[0][s]) and torch.equal(a.c[s], before[1][s])
        assert torch.equal(a.pred_proj[s], before[2][s])
    torch.cuda.synchronize()


@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
def test_compact_mode_gives_the_same_outputs(cuda, dt):
    """Compact mode (per iteration, a device list of the streams that emitted a
    token; the next symbol's joint and the LSTM / projection launches run over
    it) against the tile-by-tile launches: tokens and state bit for bit, over
    direct launches and graph replays (the lists and their counts are reset
    inside the recording), 2- and 14-frame steps, ragged lengths."""
    pred, joint, _ = _model(1026, 512, 2, dt, cuda, seed=12)
    S, B = 80, 70
    rng = np.random.default_rng(5)
    slots = rng.permutation(S)[:B]
    a = GreedyDecoder(pred, joint, blank_id=1026, num_slots=S)
    b = GreedyDecoder(pred, joint, blank_id=1026, num_slots=S)
    a.compact, b.compact = -1, 1
    a.reset_slot(slots)
    b.reset_slot(slots)
    n_tok = 0
    for step in range(8):
        T = 14 if step % 4 == 3 else 2
        enc = torch.randn(B, T, 512, generator=torch.Generator().manual_seed(100 + step)).to(dt).to(cuda)
        lens = rng.integers(0, T + 1, B)
        graph = step % 2 == 1
        ta = a.decode(slots, enc, lens, frame_tokens=True, graph=graph)
        tb = b.decode(slots, enc, lens, frame_tokens=True, graph=graph)
        assert ta == tb, f"step {step}"
        assert torch.equal(a.h, b.h) and torch.equal(a.c, b.c) and torch.equal(a.pred_proj, b.pred_proj)
        n_tok += sum(len(t) for fr in ta for t in fr)
    assert n_tok > 50, n_tok  # tokens were emitted, so the lists were exercised
    torch.cuda.synchronize()


def test_pending_results_match_blocking_calls(cuda):
    """decode(graph=True, wait=False) returns before the tokens are copied back;
    its results, consumed right away, one call later, after their buffer comes
    round again (built then) or at the end, equal the blocking calls' results,
    and the state after each step is the same."""
    dt = torch.float16
    pred, joint, _ = _model(1026, 512, 1, dt, cuda, seed=13)
    a = GreedyDecoder(pred, joint, blank_id=1026, num_slots=12)
    b = GreedyDecoder(pred, joint, blank_id=1026, num_slots=12)
    slots = np.array([3, 8, 0, 11, 5, 6, 1])
    a.reset_slot(slots)
    b.reset_slot(slots)
    rng = np.random.default_rng(4)
    want, pending = [], []
    for step in range(7):
        enc = torch.randn(7, 2, 512, generator=torch.Generator().manual_seed(50 + step)).to(dt).to(cuda)
        lens = rng.integers(0, 3, 7).astype(np.int32)  # int32: the decoder may take it as it is
        want.append(a.decode(slots, enc, lens, frame_tokens=True, graph=True))
        pending.append(b.decode(slots, enc, lens, frame_tokens=True, graph=True, wait=False))
        lens[:] = 0  # the caller's array may change; the pending result kept its own
        if step == 2:
            assert pending[2].result() == want[2]  # right away
        if step == 4:
            assert pending[3].result() == want[3]  # one call later
        torch.cuda.synchronize()
        assert torch.equal(a.h, b.h) and torch.equal(a.c, b.c) and torch.equal(a.pred_proj, b.pred_proj)
    assert [p.result() for p in pending] == want  # the rest at the end (0, 1 built when their buffer came round)
    assert sum(len(t) for w in want for s_ in w for t in s_) > 5


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("layers,vocab,streams", [(1, 130, 33), (2, 70, 5), (1, 127, 140), (1, 90, 600)])
def test_packed_weights_give_the_plain_ones(cuda, dtype, layers, vocab, streams):
    """Weights in operand order against the plain layouts, tile by tile and in
    compact mode, and the mode the library picks by batch size: the same tokens and
    state bits; a vocabulary that fills no whole tile, batches on both sides of the
    line for compact mode."""
    from parakeet_amd.modules.decoder import GreedyDecoder, Joiner, Predictor

    torch.manual_seed(layers * 100 + vocab)
    with torch.device(cuda):
        pred, joint = Predictor(640, 640, layers, vocab), Joiner(512, 640, 640, num_classes=vocab)
    joint.joint_net[-1].weight.data.mul_(4.0)
    joint.joint_net[-1].bias.data[vocab] += 1.0
    pred, joint = pred.to(dtype).eval().requires_grad_(False), joint.to(dtype).eval().requires_grad_(False)
    x = torch.randn(3, streams, 2, 512, device=cuda).to(dtype)
    slots = np.random.default_rng(0).permutation(streams)
    results = []
    for mode in ("packed", "plain", "compact", "by size"):
        dec = GreedyDecoder(pred, joint, blank_id=vocab, num_slots=streams)
        if mode == "plain":
            for k in ("w_ih", "w_hh", "w_pred", "w_out"):
                delattr(dec, k + "_packed")
        dec.compact = {"compact": 1, "by size": 0}.get(mode, -1)
        dec.reset_slot(slots)
        toks = [[list(t) for t in dec.decode(slots, x[i], lengths=None if i else [1 + (b % 2) for b in range(streams)])] for i in range(3)]
        results.append((toks, dec.h.clone(), dec.c.clone(), dec.pred_proj.clone()))
    assert sum(len(t) for step in results[0][0] for t in step) > 0
    for other in results[1:]:
        assert other[0] == results[0][0]
        for a, b in zip(results[0][1:], other[1:]):
            assert torch.equal(a, b)
