"""The decoder's one-launch token step (scope_decoder_step) against the
layer-by-layer step on the same state.  Both round the same bf16 values at the
same places and differ in the order of their fp32 sums only, so single bf16
results may round to a neighbour and travel on: the bar on logits (of scale
15 ± 0.5) is the one of the token loop against the prefill, 5e-2, and on the
caches 2^-4 (a few bf16 steps of values of order 1 to 4)."""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _model(max_len, fused=True, layers=16, window=4, budget=4, **kw):
    from scope_amd.decode import DecoderConfig, ScopeDecoder

    m = ScopeDecoder(DecoderConfig(num_layers=layers, window=window, budget=budget), max_len=max_len, device=DEV, seed=5,
                     **kw)
    if not fused:
        m._fused = lambda: None
    return m


def _close(a, b, t):
    for i, (x, y) in enumerate(zip(a.k_cache + a.v_cache, b.k_cache + b.v_cache)):
        if x is not None:  # (a NaN fails every comparison here)
            err = (x[:, :t].float() - y[:, :t].float()).abs().max().item()
            assert err <= 2.0 ** -4, f"cache {i}: difference {err:.3e}"
    for i, (x, y) in enumerate(zip(a.kbar, b.kbar)):
        if x is not None:
            err = (x - y).abs().max().item()
            assert err <= 2.0 ** -4, f"key means {i}: difference {err:.3e}"


def _logits_close(a, b, what):
    """Elementwise 5e-2, and 3e-2 of the spread about the logits' middle (15) in
    the 2-norm: bf16 values that round to a neighbour at sixteen layers' places
    show up to 1e-2 there.  Returns the largest difference."""
    assert bool(torch.isfinite(a).all()) and bool(torch.isfinite(b).all()), what
    d, rel = (a - b).abs().max().item(), ((a - b).norm() / (b - 15).norm()).item()
    assert d <= 5e-2 and rel <= 3e-2, f"{what}: {d:.3e}, {rel:.3e} of the spread"
    return d, rel


@pytest.mark.parametrize("layers,window,budget,T0,n", [(16, 4, 4, 256, 133), (8, 2, 1, 128, 9), (6, 20, 11, 1152, 5)])
def test_step_equals_layer_by_layer(layers, window, budget, T0, n):
    """A block opening, its steps (a document opens inside), its closing and
    the next opening; the smallest and the widest lists (4 and 32 entries)."""
    print(f"one-launch step: {layers} layers, lists of {window + budget + 1}, {n} steps", flush=True)
    g = torch.Generator().manual_seed(9)
    toks = torch.randint(0, 50256, (T0 + n,), generator=g)
    toks[[T0 // 2, T0 + 4]] = 50256
    one, ref = (_model(T0 + 256, f, layers, window, budget, use_graph=False) for f in (True, False))
    assert one._fused() is not None
    for m in (one, ref):
        m.prefill(toks[:T0])
    worst = (0.0, 0.0)
    for s in range(n):
        worst = max(worst, _logits_close(one.step(toks[T0 + s]), ref.step(toks[T0 + s]), f"step {s}"))
    assert torch.equal(one.docs, ref.docs) and torch.equal(one.tokens, ref.tokens)
    assert int(one._t_dev) == int(ref._t_dev) == T0 + n
    _close(one, ref, T0 + n)
    print(f"  max logit difference {worst[0]:.3e}, there {worst[1]:.3e} of the spread", flush=True)


def test_token_outside_the_vocabulary_and_other_sizes():
    """A device token outside the vocabulary leaves tokens and docs as they
    are and enters as a zero row, as in the layer-by-layer step; other widths
    are not served."""
    one, ref = (_model(256, f, 6, use_graph=False) for f in (True, False))
    toks = torch.randint(0, 50256, (130,), generator=torch.Generator().manual_seed(1))
    bad = torch.tensor([60000], device=DEV)
    for m in (one, ref):
        m.prefill(toks[:128])
        m.step(toks[128])
    _logits_close(one.step(bad), ref.step(bad), "bad token")
    assert torch.equal(one.docs, ref.docs) and torch.equal(one.tokens, ref.tokens)
    from scope_amd.decode import DecoderConfig, ScopeDecoder

    small = ScopeDecoder(DecoderConfig(num_layers=6, num_heads=2, model_dim=256), max_len=256, device=DEV, seed=1)
    assert small._fused() is None


def test_two_decoders_on_two_streams():
    """Steps of two decoders queued on two streams at the same time (each
    needs all of its workgroups resident) give what they give one by one."""
    toks = torch.randint(0, 50256, (160,), generator=torch.Generator().manual_seed(2)).to(DEV)
    ms = [_model(256, True, 6, use_graph=False) for _ in range(2)]
    want = []
    for rnd in range(2):
        outs = [[], []]
        for m in ms:
            m.prefill(toks[:128])
            m.step(toks[128:129])
        torch.cuda.synchronize()
        streams = [torch.cuda.Stream(), torch.cuda.Stream()] if rnd else [torch.cuda.current_stream()] * 2
        for s in range(129, 155):
            for i, m in enumerate(ms):
                with torch.cuda.stream(streams[i]):
                    outs[i].append(m.step(toks[s:s + 1]))
        torch.cuda.synchronize()
        if rnd == 0:
            want = outs
    for i in range(2):
        assert all(torch.equal(a, b) for a, b in zip(outs[i], want[i])), f"decoder {i}"


def test_expired_wait_gives_nan_and_raises():
    """With the status word set (as a wait that lasted too long leaves it) the
    kernel ends at once with NaN rows; with the host's copy set, step raises."""
    m = _model(256, True, 6, use_graph=False)
    toks = torch.randint(0, 50256, (140,), generator=torch.Generator().manual_seed(3))
    m.prefill(toks[:128])
    m.step(toks[128])
    work = m._fused()[2]
    work[4:8].copy_(torch.tensor([1, 0, 0, 0], dtype=torch.uint8, device=DEV))
    assert bool(torch.isnan(m.step(toks[129])).all())
    work[4:8].zero_()
    m.prefill(toks[:128])
    m.step(toks[128])
    assert bool(torch.isfinite(m.step(toks[129])).all())
    m._step_status[0] = 1
    with pytest.raises(RuntimeError, match="waited too long"):
        m.step(toks[130])
    # the next request starts over with a workspace of its own
    m.prefill(toks[:128])
    m.step(toks[128])
    assert bool(torch.isfinite(m.step(toks[129])).all())


def test_replaced_weights_of_another_layout():
    """A weight replaced in place of its memory by one of another layout is
    seen: the one-launch step serves contiguous rows only."""
    m = _model(256, True, 6, use_graph=False)
    assert m._fused() is not None
    w = m.layers[0]["mlp_fc"]
    m.layers[0]["mlp_fc"] = torch.as_strided(w, w.shape, (1, w.shape[0]))  # the same address
    assert m._fused() is None
    m.layers[0]["mlp_fc"] = w
    assert m._fused() is not None


def test_token_outside_the_vocabulary_stays_in_its_document():
    """After documents have opened, such a token (the padded columns of the
    logits have ids past the vocabulary) attends to the document its position
    carries, as in the layer-by-layer step, and its k and v rows, which later
    tokens read, are the same."""
    one, ref = (_model(384, f, 6, use_graph=False) for f in (True, False))
    toks = torch.randint(0, 50256, (140,), generator=torch.Generator().manual_seed(4))
    toks[[40, 100]] = 50256
    bad = torch.tensor([50280], device=DEV)
    for m in (one, ref):
        m.prefill(toks[:128])
        m.step(toks[128])
    for s in range(129, 135):
        tok = bad if s == 131 else toks[s]
        _logits_close(one.step(tok), ref.step(tok), f"position {s}")
    assert torch.equal(one.docs, ref.docs)
    _close(one, ref, 135)


@pytest.mark.parametrize("where", ["query", "hidden", "key", "value"])
def test_nan_reaches_the_logits(where):
    """A NaN inside a layer (an expired wait goes on with one) is in every
    logit: a head's whole query (all scores NaN), one hidden unit of the MLP,
    one visible key or value (some scores or products NaN)."""
    m = _model(256, True, 6, use_graph=False)
    toks = torch.randint(0, 50256, (140,), generator=torch.Generator().manual_seed(6))
    m.prefill(toks[:128])
    m.step(toks[128])
    assert bool(torch.isfinite(m.step(toks[129])).all())
    if where == "query":
        m.layers[2]["qkv"][128:256] = float("nan")  # head 1
    elif where == "hidden":
        m.layers[2]["mlp_fc"][77] = float("nan")
    else:
        (m.k_cache if where == "key" else m.v_cache)[2][1, 60] = float("nan")
    assert bool(torch.isnan(m.step(toks[130])).all())


@pytest.mark.parametrize("which", ["every v cache", "one k cache", "longer caches", "one list", "one list of 64 bits"])
def test_caches_and_lists_of_another_layout(which):
    """Caches whose rows lie otherwise, or are more, in all layers are served; one that
    differs from the others, or a list that is not contiguous int32, leaves the
    step to the layer-by-layer kernels, with the same logits."""
    ms = [_model(256, f, 6, use_graph=False) for f in (True, False)]
    toks = torch.randint(0, 50256, (140,), generator=torch.Generator().manual_seed(8))
    if which == "one list of 64 bits":
        ms = ms[:1]
    for m in ms:
        if which == "every v cache":
            m.v_cache = [c if c is None else torch.zeros_like(c.transpose(0, 1).contiguous()).transpose(0, 1)
                         for c in m.v_cache]
        elif which == "longer caches":
            m.k_cache, m.v_cache = ([c if c is None else torch.zeros((8, 512, 128), dtype=c.dtype, device=DEV)
                                     for c in cs] for cs in (m.k_cache, m.v_cache))
        elif which == "one k cache":
            m.k_cache[3] = torch.zeros_like(m.k_cache[3].transpose(0, 1).contiguous()).transpose(0, 1)
        elif which == "one list":
            m.list_idx[3] = torch.zeros_like(m.list_idx[3].t().contiguous()).t()
        else:
            m.list_num[3] = m.list_num[3].long()
        served = which in ("every v cache", "longer caches")
        assert (m._fused() is not None) == (served and m is ms[0])
        if which.startswith("one list"):
            return
        m.prefill(toks[:128])
    for s in range(128, 134):
        a, b = (m.step(toks[s]) for m in ms)
        _logits_close(a, b, f"position {s}")
        assert served or torch.equal(a, b)
    _close(*ms, 134)


@pytest.mark.parametrize("what,fused", [("weight", True), ("cache", True), ("lists", True), ("scale", True),
                                        ("lambdas", True), ("vlam in place", True), ("data", True), ("weight", False), ("vlam", False),
                                        ("lm_head", False)])
def test_replays_see_what_was_replaced(what, fused):
    """After a capture, a step inside a block uses the decoder's tensors and
    numbers of that moment, as an eager step does."""
    ms = [_model(256, fused, 6, use_graph=g) for g in (True, False)]
    toks = torch.randint(0, 50256, (150,), generator=torch.Generator().manual_seed(10))
    for m in ms:
        m.layers[2]["vlam"] = [0.5, 0.5]
        m.prefill(toks[:128])
    for s in range(128, 134):
        a, b = (m.step(toks[s]) for m in ms)
    assert ms[0]._graph is not None and torch.equal(a, b)
    old = []
    for m in ms:
        lay = m.layers[2]
        old.append((lay["mlp_fc"], m.k_cache[1], m.list_idx[1], m.lm_head))
        if what == "weight":
            lay["mlp_fc"] = -lay["mlp_fc"]
        elif what == "data":
            lay["mlp_fc"].data = -lay["mlp_fc"]
        elif what == "cache":
            m.k_cache[1] = -m.k_cache[1]
        elif what == "lists":
            m.list_num[1] = torch.zeros_like(m.list_num[1])
        elif what == "scale":
            m.cfg.attn_scale = 0.5
        elif what == "vlam":
            lay["vlam"] = (0.25, -0.5)
        elif what == "vlam in place":
            lay["vlam"][0] = 0.25
        elif what == "lambdas":
            lay["lambdas"] = (0.5, 1.0)
        else:
            m.lm_head = -m.lm_head
    for s in range(134, 139):
        a, b = (m.step(toks[s]) for m in ms)
        assert torch.equal(a, b), f"position {s}"
    _close(*ms, 139)


def test_table_and_workspace_belong_to_the_callers_stream():
    """They are used on the caller's stream from then on: allocated on the
    warm-up's side stream, their memory could go to new tensors of that stream
    while a step still used it."""
    m = _model(256, True, 6, use_graph=True)
    toks = torch.randint(0, 50256, (140,), generator=torch.Generator().manual_seed(11))
    m.prefill(toks[:128])
    caller = torch.cuda.Stream()
    caller.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(caller):
        for s in range(128, 133):
            m.step(toks[s])
    torch.cuda.synchronize()
    streams = {}
    for seg in torch.cuda.memory_snapshot():
        for t in m._step_table[1:]:
            if seg["address"] <= t.data_ptr() < seg["address"] + seg["total_size"]:
                streams[t.data_ptr()] = seg["stream"]
    assert list(streams.values()) == [caller.cuda_stream] * 2


@pytest.mark.parametrize("use_graph", [False, True])
def test_generate_raises_after_an_expired_wait(use_graph):
    """The last step of a request has no step after it: generate itself says
    that a wait expired (the status preset on the device, as such a wait
    leaves it), instead of the token 0 that all-NaN logits give."""
    m = _model(256, True, 6, use_graph=use_graph)
    toks = torch.randint(0, 50256, (140,), generator=torch.Generator().manual_seed(3))
    m.prefill(toks[:128])
    assert bool((m.generate(6, 5) >= 0).all())
    m._fused()[2][4:8].copy_(torch.tensor([1, 0, 0, 0], dtype=torch.uint8, device=DEV))
    with pytest.raises(RuntimeError, match="waited too long"):
        m.generate(1, 5)
    m.prefill(toks[:128])
    assert m.generate(6, 5).numel() == 6


@pytest.mark.parametrize("layers,window,budget", [(6, 4, 4), (16, 4, 4), (6, 20, 11)])
def test_step_on_some_of_its_workgroups(layers, window, budget):
    """A step that starts with some of its workgroups (no more launched, so that
    the wait for the rest ends at its limit; with a limit of 0 the launched
    ones that come later leave) gives the same bits as one on all 256."""
    toks = torch.randint(0, 50256, (1152 + 24,), generator=torch.Generator().manual_seed(7)).to(DEV)
    toks[40] = 50256
    want = caches = None
    for some in (False, True):
        m = _model(1280, True, layers, window, budget, use_graph=False)
        m.prefill(toks[:1152])
        m.step(toks[1152:1153])
        prm, _, work = m._fused()
        got, seen = [], []
        for s in range(1153, 1176):
            launched = (0, 1, 2, 7, 71, 128, 250, 255)[s % 8] if some else 0
            limit = 0 if some and s >= 1168 else 20_000
            prm.workgroups, prm.gang_ticks = launched, limit
            got.append(m.step(toks[s:s + 1]))
            word = int(work[8:12].cpu().view(torch.int32)) & 0xFFFFFFFF
            seen.append((word >> 16) & 0x7FFF if word >> 31 else word)
            assert seen[-1] == (launched or 256) or (limit == 0 and 0 < seen[-1] <= (launched or 256))
        if some:
            print(f"  workgroups of the steps: {seen}", flush=True)
            assert all(torch.equal(a, b) for a, b in zip(got, want))
            assert all(x is None or torch.equal(x, y) for x, y in zip(m.k_cache + m.v_cache, caches))
            assert int(m._t_dev) == 1176 and torch.equal(m.tokens[:1176], toks)
        else:
            want, caches = got, m.k_cache + m.v_cache


def test_two_threads_replaying_on_streams_of_their_own():
    """Two decoders driven by two threads (each replay takes the step lock and
    runs the step) give what each gives alone."""
    import threading

    g = torch.Generator().manual_seed(12)
    toks = [torch.randint(0, 50256, (128 + 120,), generator=g).to(DEV) for _ in range(2)]
    ms = [_model(256, True, 6, use_graph=True) for _ in range(2)]

    def request(i):
        ms[i].prefill(toks[i][:128])
        return torch.stack([ms[i].step(t) for t in toks[i][128:].split(1)])

    want = [request(i) for i in range(2)]  # the graphs are captured here
    torch.cuda.synchronize()
    got, streams = [None, None], [torch.cuda.Stream(), torch.cuda.Stream()]

    def work(i):
        with torch.cuda.stream(streams[i]), torch.no_grad():
            for _ in range(3):
                got[i] = request(i)
            streams[i].synchronize()

    threads = [threading.Thread(target=work, args=(i,), daemon=True) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(timeout=60)
    assert all(torch.equal(a, b) for a, b in zip(got, want))


_CHILD = """
import sys, torch
sys.path.insert(0, {root!r})
from tests.test_gpu_decode_step import _decode_alone
print("ready", flush=True)
sys.stdin.readline()
print(_decode_alone(int(sys.argv[1])), flush=True)
"""


def _decode_alone(seed):
    """The tokens of three short requests (a graph after the first steps)."""
    m = _model(512, True, 6, use_graph=True)
    g = torch.Generator().manual_seed(seed)
    out = []
    for _ in range(3):
        m.prefill(torch.randint(0, 50256, (128,), generator=g))
        out.append(m.generate(300, 17))
    return [t.tolist() for t in out]


def test_two_processes_on_one_device():
    """Two processes that decode on the same device at the same time (their
    steps compete for the same compute units) get what one alone gets."""
    import os
    import subprocess
    import sys

    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    want = _decode_alone(21)
    print("  alone: done", flush=True)
    child = subprocess.Popen([sys.executable, "-c", _CHILD.format(root=root), "21"], cwd=root, stdin=subprocess.PIPE,
                             stdout=subprocess.PIPE, text=True)
    try:
        assert child.stdout.readline().strip() == "ready"
        child.stdin.write("go\n")
        child.stdin.flush()
        print("  child started", flush=True)
        assert _decode_alone(21) == want
        assert child.communicate(timeout=60)[0].strip() == str(want)
        assert child.returncode == 0
    finally:
        child.kill()
