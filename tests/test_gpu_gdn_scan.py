"""The chunked varlen GDN prefill (csrc/gdn_scan.hip) where it can go wrong:
edges of the 32-token chunks, the 64-token groups and the 512-token segments,
strides without the 16-byte form, values that are not finite, graph replays.
Reference: the token-by-token recurrence in float64."""

import pytest
import torch

pytestmark = pytest.mark.gpu

H, D = 2, 128
SEG = 512


def inputs(T, dev, seed, decay=1.0):
    gen = torch.Generator().manual_seed(seed)
    r = lambda *s: torch.randn(*s, generator=gen)  # noqa: E731
    q = torch.nn.functional.normalize(r(T, H, D), dim=-1) * D ** -0.5
    k = torch.nn.functional.normalize(r(T, H, D), dim=-1)
    g = -torch.nn.functional.softplus(r(T, H)) * decay
    return [x.to(dev) for x in (q.bfloat16(), k.bfloat16(), r(T, H, D).bfloat16(),
                                torch.sigmoid(r(T, H)), g)]


def recurrence64(q, k, v, beta, g, lens):
    outs, states, o = [], [], 0
    q, k, v, beta, g = (x.double() for x in (q, k, v, beta, g))
    for n in lens:
        s = torch.zeros(H, D, D, dtype=torch.float64, device=q.device)
        for t in range(o, o + n):
            s = s * torch.exp(g[t])[:, None, None]
            d = beta[t][:, None] * (v[t] - (k[t][:, :, None] * s).sum(1))
            s = s + k[t][:, :, None] * d[:, None, :]
            outs.append((q[t][:, :, None] * s).sum(1))
        states.append(s)
        o += n
    return torch.stack(outs), torch.stack(states)


def cu_of(lens, dev):
    return torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist(), dtype=torch.int32,
                        device=dev)


def rel(x, y):
    return float((x.double() - y).norm() / y.norm())


# decay 0.003: a memory of hundreds of tokens, so that segments feel each other
@pytest.mark.parametrize("lens, decay", [
    ([31, 32, 33], 1.0), ([63, 64, 65, 1], 0.05), ([SEG - 1, SEG, SEG + 1], 0.003),
    ([2 * SEG + 33, 5, 3 * SEG], 0.003), ([40], 30.0)])
def test_lengths_vs_recurrence(pkg, dev, lens, decay):
    args = inputs(sum(lens), dev, 7 + sum(lens), decay)
    out, st = pkg.gdn_recurrent_prefill_sequential(*args, cu_of(lens, dev))
    o64, s64 = recurrence64(*args, lens)
    # out: one bf16 rounding (2^-9 at most, 2^-9.2 rms); state: fp32 sums over
    # the memory's tokens, measured at most 3.4e-7 (the token-by-token fp32
    # kernel it replaced: 1.3e-6)
    assert rel(out, o64) < 2 ** -9
    assert rel(st, s64) < 1e-6
    # the same bits alone as in the batch
    o = 0
    for b, n in enumerate(lens):
        o1, s1 = pkg.gdn_recurrent_prefill_sequential(*(x[o:o + n] for x in args))
        assert torch.equal(s1, st[b]) and torch.equal(o1, out[o:o + n])
        o += n


# walked alone (8 tokens at most), in chunks, in segments; by the token walk's own
# kernel (one and four columns a lane: from 128 sequences of two heads) and
# inside the scan kernel; more than 64 sequences: listed segments; more than 512
@pytest.mark.parametrize("lens", [
    [1, 8, 0, 3], [8] * 40, [1, 2, 7, 8] * 33, [8, 9, 1, 40], [5] * 63 + [SEG + 1],
    [3, 9] * 34 + [2 * SEG + 5, 0, SEG + 1, 8, 2 * SEG], [4] * 520, [4] * 130 + [600]])
def test_short_sequences_same_bits_by_every_route(pkg, dev, lens):
    T = sum(lens)
    args = inputs(T, dev, 17 + T, 0.2)
    cu = cu_of(lens, dev)
    into = pkg.gdn_recurrent_prefill.gdn_prefill_sequential_into
    got = []
    for hint in (None, max(lens)):
        st = torch.full((len(lens), H, D, D), float("nan"), device=dev)
        got.append((into(*args, cu, st, hint), st))
    got.append(pkg.gdn_recurrent_prefill_sequential(*args, cu))
    for out, st in got[1:]:
        assert torch.equal(out, got[0][0]) and torch.equal(st, got[0][1])
    out, st = got[0]
    o = 0
    for b, n in enumerate(lens):
        if n and (b < 8 or b > len(lens) - 8):
            o1, s1 = pkg.gdn_recurrent_prefill_sequential(*(x[o:o + n] for x in args))
            assert torch.equal(s1, st[b]) and torch.equal(o1, out[o:o + n])
        elif n == 0:
            assert not st[b].any()
        o += n
    some = [b for b, n in enumerate(lens) if 0 < n <= 9][:6]
    starts = [sum(lens[:b]) for b in some]
    rows = torch.cat([torch.arange(o, o + lens[b]) for b, o in zip(some, starts)]).to(dev)
    o64, s64 = recurrence64(*(x[rows] for x in args), [lens[b] for b in some])
    assert rel(out[rows], o64) < 2 ** -9 and rel(st[some], s64) < 1e-6


def test_short_sequences_other_strides_and_two_column_blocks(pkg, dev):
    """Walked sequences beside long ones: other strides, and 256 value columns,
    give the bits of contiguous inputs and of each half of the columns alone."""
    lens = [8, 9, 0, 1, 40, SEG + 5]
    T = sum(lens)
    q, k, v, beta, g = inputs(T, dev, 29, 0.1)
    cu = cu_of(lens, dev)
    want = pkg.gdn_recurrent_prefill_sequential(q, k, v, beta, g, cu)
    wide = torch.zeros(T, H, 2 * D, dtype=v.dtype, device=dev)
    wide[..., ::2] = v
    got = pkg.gdn_recurrent_prefill_sequential(q, k, wide[..., ::2], beta, g, cu)
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
    v2 = torch.cat([v, v.flip(0)], -1)
    out, st = pkg.gdn_recurrent_prefill_sequential(q, k, v2, beta, g, cu)
    half = pkg.gdn_recurrent_prefill_sequential(q, k, v.flip(0).contiguous(), beta, g, cu)
    for i, (o, s) in enumerate((want, half)):
        assert torch.equal(out[..., i * D:(i + 1) * D], o)
        assert torch.equal(st[..., i * D:(i + 1) * D], s)
    prompt = pkg.call_gdn_recurrent_prefill_chunked_triton
    for n in (5, 400):
        o2, s2 = prompt(*(x[:n] for x in (q, k, v2, beta, g)))
        o1, s1 = prompt(*(x[:n] for x in (q, k, v, beta, g)))
        assert torch.equal(o2[..., :D], o1) and torch.equal(s2[..., :D], s1)


# one prompt alone: walked, in one piece, at the first cut, a segment's edges
@pytest.mark.parametrize("T", [1, 8, 9, 64, 192, 193, 256, 257, 1024, 1025, 2100])
def test_prompt_alone_vs_recurrence(pkg, dev, T):
    args = inputs(T, dev, 23 + T, 0.003)
    out, st = pkg.call_gdn_recurrent_prefill_chunked_triton(*args)
    o64, s64 = recurrence64(*args, [T])
    assert out.shape == (T, H, D) and st.shape == (H, D, D)
    assert rel(out, o64) < 2 ** -9 and rel(st, s64[0]) < 1e-6
    state = torch.full((1, H, D, D), float("nan"), device=dev)
    got = pkg.gdn_recurrent_prefill.gdn_prefill_prompt_into(*args, state)
    assert torch.equal(got, out) and torch.equal(state[0], st)


@pytest.mark.parametrize("T", [7, 33, SEG + 70])
def test_other_strides_same_bits(pkg, dev, T):
    q, k, v, beta, g = inputs(T, dev, T)

    def spread(x):
        buf = torch.zeros(*x.shape[:-1], 2 * x.shape[-1], dtype=x.dtype, device=dev)
        buf[..., ::2] = x
        return buf[..., ::2]

    want = pkg.gdn_recurrent_prefill_sequential(q, k, v, beta, g)
    heads_first = [x.transpose(0, 1).contiguous().transpose(0, 1) for x in (q, k, v, beta, g)]
    wide = torch.cat([q, k, v], -1)
    views = [wide[..., :D], wide[..., D:2 * D], wide[..., 2 * D:], beta, g]
    for args in ([spread(q), spread(k), spread(v), spread(beta), spread(g)], heads_first, views):
        got = pkg.gdn_recurrent_prefill_sequential(*args)
        assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])


@pytest.mark.parametrize("what", ["v", "k", "q", "beta", "g"])
@pytest.mark.parametrize("t", [0, 40, SEG + 3])
def test_nan_stays_behind_its_token(pkg, dev, what, t):
    """A NaN at token t reaches no earlier token and no other sequence."""
    T = SEG + 64
    args = dict(zip(("q", "k", "v", "beta", "g"), inputs(2 * T, dev, 3, 0.1)))
    cu = cu_of([T, T], dev)
    want, _ = pkg.gdn_recurrent_prefill_sequential(*args.values(), cu)
    x = args[what].clone()
    if x.ndim == 3:
        x[t, 0, 5] = float("nan")
    else:
        x[t, 0] = float("nan")
    args[what] = x
    out, st = pkg.gdn_recurrent_prefill_sequential(*args.values(), cu)
    assert torch.equal(out[:t], want[:t]) and torch.equal(out[T:], want[T:])
    assert torch.equal(out[:, 1], want[:, 1]) and torch.isfinite(st[:, 1]).all()
    bad = torch.isnan(out[:T, 0].float())
    if what == "q":      # the token's own output only
        assert bad[t].all() and bad.sum() == D and torch.isfinite(st).all()
    elif what == "v":    # that column from the token on
        assert bad[t:, 5].all() and bad.sum() == T - t
        assert torch.isnan(st[0, 0, :, 5]).all() and torch.isfinite(st[0, 0, :, :5]).all()
    else:
        assert bad[t:].all() and torch.isnan(st[0, 0]).all()


def step_recurrence64(q, k, v, beta, g):
    """One sequence with out = q S_decayed + (q k) delta, the kernels' form (at
    an infinite delta it keeps a sign that q S_new, a sum over key rows of both
    signs, has not)."""
    outs = []
    q, k, v, beta, g = (x.double().cpu() for x in (q, k, v, beta, g))
    s = torch.zeros(H, D, D, dtype=torch.float64)
    for t in range(q.shape[0]):
        s = s * torch.exp(g[t])[:, None, None]
        d = beta[t][:, None] * (v[t] - (k[t][:, :, None] * s).sum(1))
        outs.append((q[t][:, :, None] * s).sum(1) + (q[t] * k[t]).sum(1)[:, None] * d)
        s = s + k[t][:, :, None] * d[:, None, :]
    return torch.stack(outs), s


def same_class(x, y):
    x, y = x.double().cpu(), y.double().cpu()
    assert torch.equal(torch.isnan(x), torch.isnan(y))
    inf = torch.isinf(y)
    assert torch.equal(torch.isinf(x), inf) and torch.equal(x[inf], y[inf])
    fine = torch.isfinite(y)
    torch.testing.assert_close(x[fine], y[fine], atol=2e-2, rtol=2e-2)   # (two bf16 roundings)


@pytest.mark.parametrize("what", ["v", "k", "q", "beta"])
@pytest.mark.parametrize("t", [0, 20, 40, SEG + 3, SEG + 63])
def test_infinity_as_in_the_recurrence(pkg, dev, what, t):
    """An infinite input gives the recurrence's infinities, signs included, at
    its own token and in the state, and changes nothing else."""
    T = SEG + 64
    args = dict(zip(("q", "k", "v", "beta", "g"), inputs(2 * T, dev, 5, 0.1)))
    cu = cu_of([T, T], dev)
    want, want_st = pkg.gdn_recurrent_prefill_sequential(*args.values(), cu)
    x = args[what].clone()
    if x.ndim == 3:
        x[t, 0, 5] = float("inf") if t % 2 else -float("inf")
    else:
        x[t, 0] = float("inf")
    args[what] = x
    out, st = pkg.gdn_recurrent_prefill_sequential(*args.values(), cu)
    o64, s64 = step_recurrence64(*(y[:T] for y in args.values()))
    same_class(out[:T], o64)
    same_class(st[0], s64)
    assert torch.equal(out[:t], want[:t]) and torch.equal(out[T:], want[T:])
    assert torch.equal(out[:, 1], want[:, 1]) and torch.equal(st[1], want_st[1])
    if what == "v":
        assert torch.isinf(out[t, 0, 5])
        keep = torch.arange(D, device=dev) != 5
        assert torch.equal(out[:, 0, keep], want[:, 0, keep])


def test_overflow_reaches_no_earlier_token(pkg, dev):
    """beta v past FLT_MAX at token 40 from finite inputs: its column alone,
    from its own token on."""
    T = 60
    q, k, v, beta, g = inputs(T, dev, 15, 0.1)
    v[40, 0, 5] = 3e38
    beta[40, 0] = 4.0
    out, st = pkg.gdn_recurrent_prefill_sequential(q, k, v, beta, g)
    o64, s64 = step_recurrence64(q, k, v, beta, g)
    fine = torch.ones(T, H, D, dtype=torch.bool)
    fine[40:, 0, 5] = False
    assert torch.equal(torch.isfinite(out).cpu(), fine)
    same_class(out.cpu()[fine], o64[fine])
    assert torch.isfinite(st[0, :, :5]).all() and torch.isfinite(st[1]).all()


def test_full_decay_and_growth(pkg, dev):
    """g = -inf clears the state; g > 0 grows it."""
    T = 100
    q, k, v, beta, g = inputs(T, dev, 11, 0.2)
    g[37] = -float("inf")
    g[64] = -1e30
    g[70:75] = 0.5
    out, st = pkg.gdn_recurrent_prefill_sequential(q, k, v, beta, g)
    o64, s64 = recurrence64(q, k, v, beta, g, [T])
    assert rel(out, o64) < 2 ** -9 and rel(st, s64[0]) < 1e-6


def test_growth_after_full_decay_brings_nothing_back(pkg, dev):
    """What a factor exp(-400) cleared stays cleared when later tokens of the
    same chunk grow the state by exp(80) (beta = 0 there: the state is zero)."""
    T = 100
    q, k, v, beta, g = inputs(T, dev, 13, 0.2)
    g[37] = -400.0
    beta[37:60] = 0.0
    g[40:42] = 40.0
    out, st = pkg.gdn_recurrent_prefill_sequential(q, k, v, beta, g)
    o64, s64 = recurrence64(q, k, v, beta, g, [T])
    assert (out[37:60] == 0).all()
    assert rel(out, o64) < 2 ** -9 and rel(st, s64[0]) < 1e-6


def test_graph_replays_and_other_stream(pkg, dev):
    lens = [SEG + 40, 77]
    args = inputs(sum(lens), dev, 5, 0.05)
    cu = cu_of(lens, dev)
    st = torch.zeros(2, H, D, D, device=dev)
    into = pkg.gdn_recurrent_prefill.gdn_prefill_sequential_into
    want, want_st = into(*args, cu, st).clone(), st.clone()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        into(*args, cu, st)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        out = into(*args, cu, st)
    for _ in range(4):
        out.zero_()
        st.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want) and torch.equal(st, want_st)
        torch.randn(1 << 20, device=dev).sum()
