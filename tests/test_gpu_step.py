"""GPU parity of the serving-loop step (parakeet_amd.step.AttentionStep): every
layer's paged attention output against the oracle, step after step, with stream
arrivals and departures (slot resets), batches that name a subset of the slots
in shuffled order, and a pre-shuffled page pool.

The oracle keeps one dense shift-buffer window per slot
(parakeet/modules/cache.py:36-45), the reference's per-stream mask loop
(parakeet/modules/encoder.py:167-227) over the batch's state scalars, and the
float64 rel-pos attention (attention.py:94-121).  Tolerance as in
test_gpu_attention.py; pages are also checked bit-exact through pk_kv_gather.
"""

import numpy as np
import pytest
import torch

from oracle import attention as oa
from oracle import masks as om
from parakeet_amd import ops, synth
from parakeet_amd.step import AttentionStep

TOL = {torch.float32: 1e-4, torch.float16: 2e-3, torch.bfloat16: 1e-2}


def _run(cuda, shape, slots, steps, seed, rows_per_lane=0, graph=False):
    print(f"\n[step] {shape.name} slots={slots} steps={steps} nr={rows_per_lane} graph={graph}", flush=True)
    T, D, Ly, L, left = shape.chunk, shape.d_model, shape.layers, shape.window, shape.left
    g = torch.Generator().manual_seed(seed)
    rng = np.random.default_rng(seed)
    qkv = [torch.zeros(slots, T, 3 * D, dtype=shape.dtype, device=cuda) for _ in range(Ly)]
    pos, _, _ = synth.relpos_inputs(shape, cuda, seed=seed)
    bu = [(torch.randn(shape.heads, shape.head_dim, generator=g) * 0.02).to(shape.dtype).to(cuda) for _ in range(Ly)]
    bv = [(torch.randn(shape.heads, shape.head_dim, generator=g) * 0.02).to(shape.dtype).to(cuda) for _ in range(Ly)]
    M = (L + shape.page_size - 2) // shape.page_size + 1
    order = rng.permutation(slots * M)
    st = AttentionStep(shape, slots, cuda, qkv, pos, bu, bv, page_order=order, rows_per_lane=rows_per_lane)
    # poison: a read of a never-written page row shows up as NaN
    st.k_pages.fill_(float("nan"))
    st.v_pages.fill_(float("nan"))

    win_k = np.zeros((slots, Ly, L, D))
    win_v = np.zeros((slots, Ly, L, D))
    proc = np.zeros(slots, dtype=np.int64)
    cl = np.zeros(slots, dtype=np.int64)
    pos64 = pos.double().cpu().numpy()
    worst = 0.0
    for step in range(steps):
        if step and step % 7 == 0:
            gone = rng.choice(slots, size=2, replace=False)
            st.reset_slots(gone)
            for s in gone:  # scheduler.py:86-91 zeroes a slot
                win_k[s] = 0
                win_v[s] = 0
                proc[s] = 0
                cl[s] = 0
        batch = rng.permutation(slots)[: max(1, slots - step % 3)]
        B = len(batch)
        frames = []
        for layer in range(Ly):
            x = torch.randn(B, T, 3 * D, generator=g).to(shape.dtype)
            qkv[layer][:B].copy_(x.to(cuda))
            frames.append(x.double().numpy())
        st.step(batch, graph=graph)
        _, mask = om.create_streaming_masks(T, cl[batch], proc[batch], T, (left, shape.right))
        for layer in range(Ly):
            q, k, v = np.split(frames[layer], 3, axis=-1)
            for b, s in enumerate(batch):  # cache.py:36-45 per slot
                for win, new in ((win_k, k[b]), (win_v, v[b])):
                    win[s, layer, :left] = win[s, layer, -left:].copy()
                    win[s, layer, left:] = new
            ref = oa.relpos_attention(
                q, win_k[batch, layer], win_v[batch, layer], pos64,
                bu[layer].double().cpu().numpy(), bv[layer].double().cpu().numpy(), mask, shape.heads,
            )
            got = st.out[layer][:B].double().cpu().numpy()
            err = float(np.abs(got - ref).max())
            worst = max(worst, err)
            assert err <= TOL[shape.dtype], f"step {step} layer {layer}: max abs err {err:.3e}"
            pages = ops.PagedKV(st.k_pages, st.v_pages, st.rows[:B], st.pool.max_pages)
            gk, gv = ops.kv_gather(pages, layer, B, L, T)
            ek = torch.from_numpy(win_k[batch, layer]).to(shape.dtype)
            ev = torch.from_numpy(win_v[batch, layer]).to(shape.dtype)
            assert torch.equal(gk.cpu(), ek) and torch.equal(gv.cpu(), ev), f"step {step} layer {layer}: pages"
        proc[batch] += T  # encoder.py:257-260
        cl[batch] = np.minimum(cl[batch] + T, left)
    torch.cuda.synchronize()
    print(f"  worst max-abs error {worst:.3e}", flush=True)


SMALL = synth.Shape("small-3layer-fp16", 3, 512, 8, dtype=torch.float16)
LARGE = synth.Shape("large-3layer-bf16", 3, 1024, 8, dtype=torch.bfloat16)
SMALL32 = synth.Shape("small-2layer-fp32", 2, 512, 8, dtype=torch.float32)


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [SMALL, LARGE, SMALL32], ids=lambda s: s.name)
def test_step_churn_matches_oracle(cuda, shape):
    _run(cuda, shape, slots=6, steps=45, seed=5)


@pytest.mark.gpu
def test_step_vector_kernel_path(cuda):
    """rows_per_lane forces the vector-ALU kernel for 16-bit types too."""
    _run(cuda, SMALL, slots=5, steps=30, seed=6, rows_per_lane=9)


@pytest.mark.gpu
def test_step_t14_chunks(cuda):
    """The real large model's att_context_size (70, 13): 14-frame chunks that
    straddle pages and several query groups per stream."""
    shape = synth.Shape("large-t14-bf16", 2, 1024, 8, right=13, dtype=torch.bfloat16)
    _run(cuda, shape, slots=4, steps=14, seed=7)


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [SMALL, LARGE], ids=lambda s: s.name)
def test_step_graph_replays_match_oracle(cuda, shape):
    """All layers recorded once in a HIP graph and replayed every step for
    batches of changing size (the live count is read on the device); between
    replays the test's own eager work runs (uploads, gathers, copies back,
    synchronizations) and every replay is checked against the oracle."""
    _run(cuda, shape, slots=6, steps=30, seed=8, graph=True)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("streams,layers,d,right", [(1, 3, 512, 1), (5, 33, 512, 0), (37, 4, 512, 1), (9, 5, 1024, 13), (130, 3, 1024, 1), (3, 2, 512, 6)])
def test_layers_in_one_launch_match_layer_by_layer(cuda, dtype, streams, layers, d, right):
    """pk_paged_relpos_attn_layers (AttentionStep's launch over every layer; past 32
    layers two launches, fp32 one by one) against one launch a layer: outputs and
    pages bit for bit, over steps that evict, with streams of several ages, and
    replayed from a graph over a smaller batch."""
    import numpy as np

    from parakeet_amd import synth
    from parakeet_amd.step import AttentionStep

    T, left = right + 1, 20
    shape = synth.Shape("layers", layers, d, 8, left=left, right=right, dtype=dtype)
    g = torch.Generator(device="cuda").manual_seed(streams + layers)
    pos = torch.randn(2 * (left + T) - 1, d, generator=g, device=cuda).to(dtype)
    bu, bv = ([torch.randn(8, d // 8, generator=g, device=cuda).to(dtype) for _ in range(layers)] for _ in range(2))
    qkv = [torch.zeros(streams, T, 3 * d, dtype=dtype, device=cuda) for _ in range(layers)]
    steps = [AttentionStep(shape, streams, torch.device("cuda", 0), qkv, pos, bu, bv) for _ in range(3)]
    for st in steps:
        st.k_pages.zero_()
        st.v_pages.zero_()
    rng = np.random.default_rng(0)
    ev = [tuple(torch.cuda.Event(enable_timing=True) for _ in range(2)) for _ in range(layers)]
    for a, b in ev:
        a.record()
        b.record()
    for i in range(left // T + 4):
        n = streams if i % 3 else max(1, streams // 2)
        slots = np.sort(rng.permutation(streams)[:n]).astype(np.int32)
        for x in qkv:
            x.copy_(torch.randn(x.shape, generator=g, device=cuda).to(dtype))
        steps[0].step(slots)
        steps[1].step(slots, events=[(a.cuda_event, b.cuda_event) for a, b in ev])  # one launch a layer
        steps[2].step(slots, graph=True)
        torch.cuda.synchronize()
        for other in steps[1:]:
            assert torch.equal(steps[0].k_pages, other.k_pages) and torch.equal(steps[0].v_pages, other.v_pages)
            for a, b in zip(steps[0].out, other.out):
                assert torch.equal(a[:n], b[:n])


def test_step_launches_on_the_stream_of_the_call(monkeypatch):
    """The upload of a step's rows and the caller's projections are on the stream
    that is current at the call; so is the launch that reads them, whichever stream
    was current when the step was built (CPU: the library replaced)."""
    import types

    import parakeet_amd.step as S

    seen, current = [], ["at construction"]
    monkeypatch.setattr(S, "lib", lambda: types.SimpleNamespace(pk_paged_relpos_attn_layers=lambda a, n, s: seen.append((n, s)) or 0))
    monkeypatch.setattr(ops, "_stream", lambda dev: (dev, current[0]))
    st = object.__new__(AttentionStep)
    st.device, st.batch, st._args, st._stream = "dev", 2, (S.AttnArgs * 3)(), ("dev", current[0])
    st.run()
    current[0] = "another"
    st.run()
    assert seen == [(3, ("dev", "at construction")), (3, ("dev", "another"))]


@pytest.mark.gpu
@pytest.mark.parametrize("graph", [False, True])
def test_steps_under_another_stream(cuda, graph):
    """Built on the default stream and stepped under another one, behind work that
    writes the projections there: outputs and pages as a step on one stream alone."""
    shape = synth.Shape("streams", 3, 512, 8, left=20, dtype=torch.float16)
    B, T, D = 5, shape.chunk, 512
    g = torch.Generator(device="cuda").manual_seed(9)
    pos = torch.randn(2 * shape.window - 1, D, generator=g, device=cuda).half()
    bias = [torch.randn(8, 64, generator=g, device=cuda).half() for _ in range(3)]
    x = torch.randn(14, 3, B, T, 3 * D, generator=g, device=cuda).half()
    big = torch.randn(4096, 4096, generator=g, device=cuda).half()
    out = []
    for stream in (torch.cuda.current_stream(), torch.cuda.Stream()):
        qkv = [torch.zeros(B, T, 3 * D, dtype=torch.float16, device=cuda) for _ in range(3)]
        st = AttentionStep(shape, B, torch.device("cuda", 0), qkv, pos, bias, bias)
        st.k_pages.zero_()
        st.v_pages.zero_()
        torch.cuda.synchronize()
        with torch.cuda.stream(stream):
            for i in range(len(x)):
                for _ in range(4):
                    big @ big  # the copies below are still to come when the step is called
                for layer in range(3):
                    qkv[layer].copy_(x[i, layer])
                st.step(np.arange(B), graph=graph)
        torch.cuda.synchronize()
        out.append([o.clone() for o in st.out] + [st.k_pages, st.v_pages])
    for a, b in zip(*out):
        assert torch.equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("right", [14, 15])
def test_layers_without_a_common_launch(cuda, dtype, right):
    """Chunks of 15 and 16 frames have no several-layer form: the one call launches
    its layers one by one, with the same bits."""
    test_layers_in_one_launch_match_layer_by_layer(cuda, dtype, 5, 3, 512, right)
