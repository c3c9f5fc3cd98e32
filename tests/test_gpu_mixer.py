"""GPU: the mixer kernels of a decoder layer against the decoder-layer oracle (``oracle/stack.py``).

The lengths are those where the GDN kernels can go wrong: one token, a chunk one short, full and one over, a ragged
last chunk; value heads per key head 1 and 4.  The oracle follows the rule token by token in float64 on the
bf16-rounded projections, so what differs is the order of fp32 sums and the bf16 rounding of
the two projections: outputs within one bf16 ulp of a projection that rounds the other way.  bf16 keeps 8 significant
bits, so an ulp of a value in [2^e, 2^(e+1)) is 2^(e-7), at most 2^-7 of the largest value.
"""
import pytest
import torch

from oracle import metrics, stack
from stack_util import oracle_layer_state, oracle_layer_weights

pytestmark = pytest.mark.gpu
TOL = 2.0 ** -7


def _gdn_model(pkg, device, key_heads, value_heads, tokens):
    base = pkg.target.small_config(("linear_attention",))
    c = type(base)(**{**vars(base), "linear_key_heads": key_heads, "linear_value_heads": value_heads})
    host = pkg.target.random_weights(c, seed=7, device="cpu", layout="portable", generate_on="cpu")
    layout = "tiled" if tokens <= 32 else "portable"
    model = pkg.target.TargetModel(pkg.target.to_device(host, device, layout=layout), capacity=96)
    return c, host, model, model.synthetic_context(5, seed=8)


@pytest.mark.parametrize("key_heads,value_heads", [(4, 16), (16, 16)])
@pytest.mark.parametrize("tokens", [1, 3, 15, 16, 17, 32, 41])
def test_gdn_layer_matches_oracle(pkg, device, tokens, key_heads, value_heads):
    c, host, model, state = _gdn_model(pkg, device, key_heads, value_heads, tokens)
    x = torch.randn((tokens, c.hidden), generator=torch.Generator().manual_seed(tokens))
    assert pkg.ops.gdn_mixer_fits(x.to(device), state.conv[0], state.recurrent[0], **model._gdn_args(model.w.layers[0]))
    trace = {}
    _, pending = model.layer(0, x.to(device), state, trace=trace)
    lw = oracle_layer_weights(host.layers[0])
    before = oracle_layer_state(state, 0)
    normed = stack.bf16(stack.norm(x, lw["input_norm"], c.rms_eps, 1.0))
    ref = stack.gdn_layer(normed, lw, before["conv"], before["recurrent"], c)
    mid = x + ref["out"]
    print(f"gdn T={tokens} {key_heads}/{value_heads}", metrics.compare(trace["mid"].cpu(), mid), flush=True)
    assert metrics.compare(trace["mid"].cpu(), mid)["max_rel"] <= TOL
    want = stack.bf16(stack.norm(trace["mid"].cpu(), lw["post_norm"], c.rms_eps, 1.0))
    assert metrics.compare(trace["moe_in"].float().cpu(), want)["max_rel"] <= TOL
    assert metrics.compare(pending.window[0].float().cpu(), ref["window"])["max_rel"] <= TOL
    for j in sorted({1, tokens // 2, tokens - 1, tokens} - {0}):
        trial = state.clone()
        model.commit(trial, pkg.target.Pending(state.position, tokens, [pending]), j)
        assert metrics.compare(trial.recurrent[0][0].cpu(), ref["states"][j].float())["max_rel"] <= TOL, j
        assert torch.equal(trial.conv[0], pending.window[:, :, j:j + 3])


def test_gdn_layer_takes_the_general_path_for_other_forms(pkg, device):
    """A conv history that is a strided view gives the result of its contiguous copy."""
    c, _, model, state = _gdn_model(pkg, device, 4, 16, 16)
    x = torch.randn((16, c.hidden), generator=torch.Generator().manual_seed(3)).to(device)
    want, _ = model.layer(0, x, state)
    state.conv[0] = state.conv[0].transpose(1, 2).contiguous().transpose(1, 2)
    assert not pkg.ops.gdn_mixer_fits(x, state.conv[0], state.recurrent[0], **model._gdn_args(model.w.layers[0]))
    got, _ = model.layer(0, x, state)
    assert metrics.compare(got.cpu(), want.cpu())["max_rel"] <= TOL


@pytest.mark.parametrize("heads,kv_heads,head_dim", [(4, 2, 128), (16, 2, 256)])
@pytest.mark.parametrize("tokens,context", [(1, 0), (1, 1), (1, 300), (2, 31), (15, 113), (16, 0), (16, 1000), (17, 40),
                                            (32, 97), (37, 0), (130, 5)])
def test_attention_layer_matches_oracle(pkg, device, tokens, context, heads, kv_heads, head_dim):
    """Lengths around the kernels' edges: row tiles of 16 (a token has heads / kv_heads rows), 32 keys a wave, 128 keys a
    workgroup, one split and many, splits past a tile's last key.  Output and K rows within one bf16 ulp (above)."""
    base = pkg.target.small_config(("full_attention",))
    c = type(base)(**{**vars(base), "heads": heads, "kv_heads": kv_heads, "head_dim": head_dim})
    host = pkg.target.random_weights(c, seed=9, device="cpu", layout="portable", generate_on="cpu")
    layout = "tiled" if tokens <= 32 else "portable"
    model = pkg.target.TargetModel(pkg.target.to_device(host, device, layout=layout), capacity=context + tokens + 3)
    state = model.synthetic_context(context, seed=10)
    state.keys[0].mul_(4.0)                         # scores of several units, so that the softmax is not flat
    before = oracle_layer_state(state, 0)
    untouched = state.keys[0][:, :, context + tokens:].clone()
    x = torch.randn((tokens, c.hidden), generator=torch.Generator().manual_seed(tokens + context))
    trace = {}
    out, pending = model.layer(0, x.to(device), state, trace=trace)
    assert pending is None and trace["mid"].dtype == torch.float32
    lw = oracle_layer_weights(host.layers[0])
    normed = stack.bf16(stack.norm(x, lw["input_norm"], c.rms_eps, 1.0))
    ref = stack.attention_layer(normed, lw, before["keys"], before["values"], context, c)
    mixer = trace["mid"].cpu() - x                  # the residual would hide it
    print(f"attention T={tokens} ctx={context} D={head_dim}", metrics.compare(mixer, ref["out"]), flush=True)
    assert metrics.compare(mixer, ref["out"])["max_rel"] <= TOL
    rows = slice(context, context + tokens)
    assert metrics.compare(state.keys[0][0, :, rows].float().cpu(), ref["keys"])["max_rel"] <= TOL
    assert metrics.compare(state.values[0][0, :, rows].float().cpu(), ref["values"])["max_rel"] <= TOL
    assert torch.equal(state.keys[0][:, :, context + tokens:], untouched)
    assert torch.equal(state.keys[0][0, :, :context].cpu(), before["keys"][:, :context])


def test_attention_layer_over_more_splits_than_lanes(pkg, device):
    """66 splits of the keys: the merge takes two of them in some lanes."""
    test_attention_layer_matches_oracle(pkg, device, 1, 8400, 16, 2, 256)


@pytest.mark.parametrize("tokens,split_down", [(1, False), (16, False), (16, True), (40, False), (260, False)])
def test_moe_with_the_residual_add(pkg, device, tokens, split_down):
    """The layer that leaves residual + output equals the layer and the add bit for bit, on every path with a combine of
    its own (verify block, its split down, the work-table kernels, the prefill tiles)."""
    layer = pkg.synthetic.moe_layer(tokens, hidden=512, inter=512, experts=16, seed=tokens)
    shared = pkg.SharedExpert(layer.shared.gate_up.to(device), layer.shared.down.to(device),
                              layer.shared.gate_weight.to(device))
    args = dict(top_k=4, router_weight=layer.router_weight.to(device), shared=shared)
    x, banks = layer.hidden.to(device), (layer.gate_up.to(device), layer.down.to(device))
    residual = torch.randn((tokens, 512), generator=torch.Generator().manual_seed(1)).to(device)
    with pkg.ops.split_down(split_down):
        want = residual + pkg.ops.moe_w4a16(x, *banks, **args)
        got = pkg.ops.moe_w4a16_add(residual, x, *banks, **args)
    assert torch.equal(got, want)
    with pytest.raises(ValueError, match="residual"):
        pkg.ops.moe_w4a16_add(residual.to(torch.bfloat16), x, *banks, **args)


def _attention_model(pkg, device, heads, kv_heads, head_dim, capacity, layout="tiled"):
    base = pkg.target.small_config(("full_attention",))
    c = type(base)(**{**vars(base), "heads": heads, "kv_heads": kv_heads, "head_dim": head_dim})
    return c, pkg.target.TargetModel(pkg.target.random_weights(c, seed=9, device=device, layout=layout), capacity=capacity)


def _mixer_and_general(model, x, state):
    """The residual after the mixer, from the kernels and from the PyTorch form of the same layer."""
    lw, eps = model.w.layers[0], model.config.rms_eps
    trace, other = {}, state.clone()
    model.layer(0, x, state, trace=trace)
    normed = (x * (x.square().mean(-1, keepdim=True) + eps).rsqrt() * (lw.input_norm + 1)).to(torch.bfloat16)
    general = x + model._attention(normed, lw, other.keys[0], other.values[0], other.position).float()
    return trace["mid"], general


@pytest.mark.parametrize("tokens,context,stretch", [
    (1, 896, None), (1, 1920, None),         # the last split holds the token's own key alone
    (1, 300, (128, 256)), (16, 1000, (128, 256)), (16, 1000, (640, 704)),     # whole splits and whole key steps
    (5, 40, (32, 33)),
])
def test_attention_keeps_a_nan_key(pkg, device, tokens, context, stretch):
    """A NaN in a visible key makes the softmax of the rows that see it NaN, wherever the key falls: a split, or a
    wave's part of one, in which every score is NaN is not one without keys."""
    c, model = _attention_model(pkg, device, 16, 2, 256, context + tokens + 3)
    state = model.synthetic_context(context, seed=10)
    if stretch is None:
        model.w.layers[0].k_norm[3] = float("nan")       # the block's own K rows
    else:
        state.keys[0][:, :, stretch[0]:stretch[1], 7] = float("nan")
    x = torch.randn((tokens, c.hidden), generator=torch.Generator().manual_seed(5)).to(device)
    got, general = _mixer_and_general(model, x, state)
    assert torch.isnan(general).all() and torch.isnan(got).all()


@pytest.mark.parametrize("kv_heads,group", [(4, 1), (4, 3)])
def test_attention_over_an_infinite_key(pkg, device, kv_heads, group):
    """A key that scores -inf has weight 0; one that scores +inf makes the row NaN, as in the softmax."""
    c, model = _attention_model(pkg, device, kv_heads * group, kv_heads, 128, 320, layout="portable")
    lw = model.w.layers[0]
    x = torch.randn((1, c.hidden), generator=torch.Generator().manual_seed(6)).to(device)
    state = model.synthetic_context(300, seed=10)
    want, _ = _mixer_and_general(model, x, state.clone())
    normed = (x * (x.square().mean(-1, keepdim=True) + c.rms_eps).rsqrt() * (lw.input_norm + 1)).to(torch.bfloat16)
    q = pkg.ops.qlinear(normed, lw.mixer_in)[0, :2 * c.heads * 128].float().view(kv_heads, group, 256)[..., 64:128]
    same = (q > 0).all(1) | (q < 0).all(1)               # a feature past the rotary ones in which a KV head's queries agree
    assert bool(same.any(1).all())
    feature = same.float().argmax(1)
    sign = q[:, 0].gather(1, feature[:, None])[:, 0].sign() * (lw.q_norm[64 + feature] + 1).sign()
    for scores, key in ((-1, 17), (-1, 299), (1, 17)):
        bad = state.clone()
        for h in range(kv_heads):
            bad.keys[0][0, h, key, 64 + feature[h]] = scores * sign[h] * float("inf")
        got, general = _mixer_and_general(model, x, bad)
        if scores > 0:
            assert torch.isnan(general).all() and torch.isnan(got).all()
        else:
            assert torch.isfinite(general).all() and not torch.equal(general, want)
            assert metrics.compare(got.cpu() - x.cpu(), general.cpu() - x.cpu())["max_rel"] <= TOL


@pytest.mark.parametrize("name", ["a_log", "dt_bias", "conv", "gdn_norm", "input_norm", "post_norm", "state"])
def test_gdn_layer_keeps_gradients(pkg, device, name):
    """Where a weight or the state asks for a gradient the PyTorch form runs, whose state and outputs carry it."""
    c, _, model, state = _gdn_model(pkg, device, 4, 16, 8)
    lw = model.w.layers[0]
    leaf = state.recurrent[0] if name == "state" else getattr(lw, name)
    leaf.requires_grad_()
    x = torch.randn((8, c.hidden), generator=torch.Generator().manual_seed(3)).to(device)
    args = model._gdn_args(lw)
    assert not pkg.ops.gdn_mixer_fits(x, state.conv[0], state.recurrent[0], **args)
    assert pkg.ops.gdn_mixer_plain(x, state.conv[0], state.recurrent[0], **args) is None
    _, pending = model.layer(0, x, state)
    assert pending.chunks[0].state.requires_grad == (name in ("a_log", "dt_bias", "conv", "state"))
    model.commit(state, pkg.target.Pending(5, 8, [pending]), 3)
    assert state.recurrent[0].requires_grad == (name in ("a_log", "dt_bias", "conv", "state"))
    with torch.no_grad():
        assert pkg.ops.gdn_mixer_plain(x, state.conv[0], state.recurrent[0].detach(), **args) is not None


@pytest.mark.parametrize("name", ["q_norm", "k_norm", "input_norm", "post_norm"])
def test_attention_layer_keeps_gradients(pkg, device, name):
    c, model = _attention_model(pkg, device, 4, 2, 128, 32)
    state, lw = model.synthetic_context(9, seed=4), model.w.layers[0]
    getattr(lw, name).requires_grad_()
    x = torch.randn((8, c.hidden), generator=torch.Generator().manual_seed(3)).to(device)
    assert model._attention_kernels(x, lw, state.keys[0], state.values[0], 9) is None
    model.layer(0, x, state)
    assert state.keys[0].requires_grad == (name == "k_norm")


@pytest.mark.parametrize("kind", ["linear_attention", "full_attention"])
def test_layer_and_final_norm_keep_forward_tangents(pkg, device, kind):
    """A forward-mode tangent of the residual goes through the residual adds and the final norm."""
    import torch.autograd.forward_ad as fwd
    c = pkg.target.small_config((kind,))
    model = pkg.target.TargetModel(pkg.target.random_weights(c, seed=3, device=device), capacity=80)
    x, v = (torch.randn((8, c.hidden), device=device) for _ in range(2))
    with torch.no_grad(), fwd.dual_level():
        dual = fwd.make_dual(x, v)
        hidden, _ = model.layer(0, dual, model.synthetic_context(9, seed=4))
        assert torch.equal(fwd.unpack_dual(hidden).tangent, v)
        out = model.forward_hidden(dual, model.synthetic_context(9, seed=4), top1=False)
        assert fwd.unpack_dual(out.hidden).tangent is not None


def test_moe_residual_add_keeps_gradients(pkg, device):
    layer = pkg.synthetic.moe_layer(4, hidden=512, inter=512, experts=16, seed=1)
    x, banks = layer.hidden.to(device), (layer.gate_up.to(device), layer.down.to(device))
    args = dict(top_k=4, router_weight=layer.router_weight.to(device))
    residual = torch.randn((4, 512), device=device)
    want = pkg.ops.moe_w4a16_add(residual, x, *banks, **args)
    got = pkg.ops.moe_w4a16_add(residual.requires_grad_(), x, *banks, **args)
    assert got.requires_grad and torch.equal(got, want)


@pytest.mark.parametrize("top_k", [True, 4.0])
def test_moe_residual_add_refuses_other_counts(pkg, device, top_k):
    """As moe_w4a16 does: an int, and no bool."""
    layer = pkg.synthetic.moe_layer(4, hidden=512, inter=512, experts=16, seed=1)
    with pytest.raises(ValueError, match="top_k must be an int"):
        pkg.ops.moe_w4a16_add(torch.zeros((4, 512), device=device), layer.hidden.to(device), layer.gate_up.to(device),
                              layer.down.to(device), top_k=top_k, router_weight=layer.router_weight.to(device))


@pytest.mark.parametrize("kind", ["linear_attention", "full_attention"])
def test_a_refused_projection_leaves_the_cache_as_it_was(pkg, device, kind, monkeypatch):
    """Tiled K = 4096 above 32 rows has no kernel: the layer is refused, once, before anything is launched or written."""
    base = pkg.target.small_config((kind,))
    c = type(base)(**{**vars(base), "heads": 16, "head_dim": 256, "linear_key_heads": 16, "linear_value_heads": 32})
    model = pkg.target.TargetModel(pkg.target.random_weights(c, seed=3, device=device, layout="tiled"), capacity=80)
    state = model.synthetic_context(9, seed=4)
    before = state.clone()
    monkeypatch.setattr(pkg._lib, "call", None)          # the Python form is not tried
    with pytest.raises(pkg._lib.DflashError, match="tiled"):
        model.layer(0, torch.randn((40, c.hidden), device=device), state)
    for a, b in zip(state.keys + state.values, before.keys + before.values):
        assert (a is None and b is None) or torch.equal(a, b)


def _signs(tokens, width, seed, device):
    """A residual of +-1: with input norm weights of 0 its bf16 norm is itself in any order of the sum, so the projection
    a mixer computes is known bit for bit."""
    return (torch.randint(0, 2, (tokens, width), generator=torch.Generator().manual_seed(seed)) * 2.0 - 1.0).to(device)


def _rel(a, b):
    return ((a.double() - b).norm() / b.norm()).item()


@pytest.mark.parametrize("key_heads,value_heads", [(4, 16), (16, 16)])
@pytest.mark.parametrize("tokens", [1, 15, 16, 48, 49, 64, 65, 97, 131])
def test_gdn_kernels_keep_fp32(pkg, device, tokens, key_heads, value_heads):
    """Outputs, writes, keys, log decays and states of every chunk, and commits inside each, against the rule token by
    token in 64 bits on the same bf16 projection.  More than three chunks: the state kernel's operand sets and its
    writing waves come round again.  Sums of 128 products in fp32, each 2^-24 off a running sum, and the state carried
    over chunks: observed up to 3e-7 of the norm; bound 2e-6 (an operand rounded to bf16 gives 2e-3)."""
    c, _, model, state = _gdn_model(pkg, device, key_heads, value_heads, tokens)
    lw = model.w.layers[0]
    lw.input_norm.zero_()
    x = _signs(tokens, c.hidden, tokens, device)
    _, pending = model.layer(0, x, state)
    kw, vw, hv = 128 * key_heads, 128 * value_heads, value_heads
    proj = pkg.ops.qlinear(x.to(torch.bfloat16), lw.mixer_in)
    qkv, z, b, a = proj.split((2 * kw + vw, vw, hv, hv), dim=-1)
    assert torch.equal(pending.window[0, :, 3:], qkv.t()) and torch.equal(pending.window[0, :, :3], state.conv[0][0])
    window, taps = pending.window[0].double(), lw.conv[:, 0].double()
    mixed = torch.nn.functional.silu(sum(window[:, i:i + tokens] * taps[:, i:i + 1] for i in range(4))).t()
    q, k, v = (m.reshape(tokens, -1, 128) for m in mixed.split((kw, kw, vw), dim=-1))
    q, k = (m * (m.square().sum(-1, keepdim=True) + 1e-6).rsqrt() for m in (q, k))
    q, k = (m.repeat_interleave(value_heads // key_heads, dim=1) for m in (q * 128 ** -0.5, k))
    beta = torch.sigmoid(b.double())
    g = -torch.exp(lw.a_log.double()) * torch.nn.functional.softplus(a.double() + lw.dt_bias.double())
    s, outs, writes, states = state.recurrent[0][0].double(), [], [], []
    for t in range(tokens):
        s = s * g[t].exp()[:, None, None]
        u = beta[t][:, None] * (v[t] - (k[t][:, None, :] @ s)[:, 0])
        s = s + k[t][:, :, None] * u[:, None, :]
        outs.append((q[t][:, None, :] @ s)[:, 0])
        writes.append(u)
        states.append(s)
    worst = {}
    assert len(pending.chunks) == (tokens + 15) // 16
    for i, ch in enumerate(pending.chunks):
        r = slice(16 * i, min(16 * i + 16, tokens))
        for name, got, want in (("out", ch.out, torch.stack(outs[r], 1)), ("u", ch.u, torch.stack(writes[r], 1)),
                                ("keys", ch.keys, k[r].transpose(0, 1)), ("cum", ch.cum, g[r].cumsum(0).t()),
                                ("state", ch.state, states[r.stop - 1])):
            assert got.shape == want[None].shape, (name, i)
            worst[name] = max(worst.get(name, 0.0), _rel(got[0], want))
            assert worst[name] <= 2e-6, (name, i, worst[name])
        for j in sorted({r.start + 1, (r.start + r.stop) // 2 + 1, r.stop} & set(range(1, tokens + 1))):
            trial = state.clone()
            model.commit(trial, pkg.target.Pending(state.position, tokens, [pending]), j)
            error = _rel(trial.recurrent[0][0], states[j - 1])
            # the log decays a commit starts from are held in fp32, each 2^-24 |G| off
            assert error <= 2e-6 + 2.0 ** -23 * ch.cum.abs().max().item(), (j, error)
            worst["commit"] = max(worst.get("commit", 0.0), error)
            assert torch.equal(trial.conv[0], pending.window[:, :, j:j + 3])
    print(f"gdn fp32 T={tokens} {key_heads}/{value_heads}", {n: f"{e:.1e}" for n, e in worst.items()}, flush=True)


def _parts(x, n):
    """The leading ``n`` bf16 parts of ``x``, summed: what a product that takes only those sees."""
    total = torch.zeros_like(x)
    for _ in range(n):
        total = total + (x - total).to(torch.bfloat16).to(x.dtype)
    return total


@pytest.mark.parametrize("heads,kv_heads,head_dim,partial", [(4, 2, 128, 0.25), (12, 4, 128, 1.0), (20, 4, 128, 0.5),
                                                             (16, 2, 256, 0.25)])
@pytest.mark.parametrize("tokens,context", [(1, 300), (7, 1000), (16, 2000), (40, 57)])
def test_attention_kernels_keep_fp32(pkg, device, tokens, context, heads, kv_heads, head_dim, partial):
    """The gated output against attention in 64 bits on the same bf16 projection and cache, through an output projection
    that is the identity (scales of 0 but for the group of the diagonal, so that a value meets the rounding of 128 others
    only; the oracle's output goes through the same projection): the share of bf16 values that come out otherwise.  Query
    heads per KV head also such that a row tile of 16 begins inside a token.  An error e of a value v flips its bf16
    rounding with probability e 2^8 / |v|: 7e-7 of the norm, at values down to a fiftieth of it, a thousandth of them, and a
    flip in turn moves the projection's fp32 rounding of its 127 neighbours, a few of which flip: observed up to 4e-3
    (one token, 1536 values), bound 6e-3.  Oracles with queries or probabilities of one bf16 part change 0.2 to 0.7 of
    the values, one with queries of two parts more than three times what the kernels do."""
    base = pkg.target.small_config(("full_attention",))
    width = heads * head_dim
    c = type(base)(**{**vars(base), "heads": heads, "kv_heads": kv_heads, "head_dim": head_dim, "hidden": width,
                      "partial_rotary": partial})
    gen = torch.Generator().manual_seed(tokens)
    in_proj = pkg.synthetic.int4_weight(gen, (2 * (heads + kv_heads) * head_dim, width)).to(device)
    out_proj = pkg.PackedW4(pkg.pack_int4(torch.eye(width, dtype=torch.int8)),
                            torch.eye(width // 128, dtype=torch.bfloat16).repeat_interleave(128, dim=0), 128).to(device)
    vec = lambda n: (torch.rand((n,), generator=gen) * 0.2 - 0.1).to(device)     # noqa: E731
    zeros = torch.zeros((width,), device=device)
    inv_freq = pkg.layers.inverse_frequencies(c.rotary_dim, c.rope_theta, device)
    q_norm, k_norm = vec(head_dim), vec(head_dim)
    keys, values = ((torch.randn((1, kv_heads, context + tokens + 3, head_dim), generator=gen) * m).to(torch.bfloat16).to(device)
                    for m in (3.0, 1.0))
    x = _signs(tokens, width, tokens + 1, device)
    mid, _ = pkg.ops.attention_mixer(x, keys, values, context, in_proj=in_proj, out_proj=out_proj, input_norm=zeros,
                                     post_norm=zeros, q_norm=q_norm, k_norm=k_norm, inv_freq=inv_freq, heads=heads,
                                     kv_heads=kv_heads, head_dim=head_dim, eps=c.rms_eps)
    proj = pkg.ops.qlinear(x.to(torch.bfloat16), in_proj).double()
    qg, k, v = proj.split((2 * heads * head_dim, kv_heads * head_dim, kv_heads * head_dim), dim=-1)
    q, gate = qg.reshape(tokens, heads, 2 * head_dim).split(head_dim, dim=-1)
    half = c.rotary_dim // 2
    angle = (torch.arange(context, context + tokens, device=device).float()[:, None] * inv_freq).double()[:, None]

    def rotated(m, weight):
        m = m * (m.square().mean(-1, keepdim=True) + c.rms_eps).rsqrt() * (weight.double() + 1)
        a, b, rest = m[..., :half], m[..., half:2 * half], m[..., 2 * half:]
        return torch.cat((a * angle.cos() - b * angle.sin(), b * angle.cos() + a * angle.sin(), rest), dim=-1)

    rows = slice(context, context + tokens)
    new_k = rotated(k.reshape(tokens, kv_heads, head_dim), k_norm).transpose(0, 1)
    assert (keys[0, :, rows] != new_k.to(torch.bfloat16)).float().mean().item() <= 2e-3
    assert torch.equal(values[0, :, rows].double(), v.reshape(tokens, kv_heads, head_dim).transpose(0, 1))
    n = context + tokens
    all_k, all_v = (m[0, :, :n].double().repeat_interleave(heads // kv_heads, dim=0) for m in (keys, values))
    q = rotated(q, q_norm).transpose(0, 1) * head_dim ** -0.5
    hidden = torch.arange(n, device=device) > torch.arange(context, n, device=device)[:, None]

    def flipped(q_parts=None, p_parts=None):
        scores = (q if q_parts is None else _parts(q, q_parts)) @ all_k.transpose(1, 2).contiguous()
        scores = scores.masked_fill(hidden, -float("inf"))
        p = (scores - scores.amax(-1, keepdim=True)).exp()
        att = (p if p_parts is None else _parts(p, p_parts)) @ all_v / p.sum(-1, keepdim=True)
        want = (att.transpose(0, 1) * torch.sigmoid(gate)).reshape(tokens, width).to(torch.bfloat16)
        return ((mid - x).to(torch.bfloat16) != pkg.ops.qlinear(want, out_proj)).float().mean().item()

    share, coarse = flipped(), [flipped(q_parts=1), flipped(p_parts=1), flipped(q_parts=2), flipped(p_parts=2)]
    print(f"attention fp32 T={tokens} ctx={context} {heads}/{kv_heads} D={head_dim}: {share:.1e}, one and two parts",
          [f"{f:.1e}" for f in coarse], flush=True)
    assert share <= 6e-3 and min(coarse[:2]) >= 0.1
    assert tokens == 1 or 2 * share <= coarse[2]


@pytest.mark.parametrize("kind", ["linear_attention", "full_attention"])
@pytest.mark.parametrize("group,scale_dtype,layout,tokens", [
    (group, dtype, layout, tokens)
    for group, dtype, layout in ((256, torch.float32, "portable"), (256, torch.float32, "tiled"), (128, torch.bfloat16, "portable"))
    for tokens in (1, 9, 32, 40) if layout == "portable" or tokens <= 32])    # tiled groups of 256 end at 32 rows
def test_mixers_over_other_banks(pkg, device, kind, tokens, group, scale_dtype, layout):
    """Groups of 256, fp32 scales and the portable layout through both mixers, against the PyTorch form on the same banks:
    both run the same projections, so what differs is fp32 sums between them and bf16 roundings that follow."""
    c = pkg.target.small_config((kind,))
    model = pkg.target.TargetModel(pkg.target.random_weights(c, seed=9, device=device, layout="portable"), capacity=96)
    lw, gen = model.w.layers[0], torch.Generator().manual_seed(group + tokens)
    for name in ("mixer_in", "mixer_out"):
        old = getattr(lw, name)
        w = pkg.synthetic.int4_weight(gen, (old.rows, old.cols), group, scale_dtype).to(device)
        setattr(lw, name, w.tiled() if layout == "tiled" else w)
    state = model.synthetic_context(21, seed=4)
    x = torch.randn((tokens, c.hidden), generator=gen).to(device)
    trace, other = {}, state.clone()
    model.layer(0, x, state, trace=trace)
    normed = (x * (x.square().mean(-1, keepdim=True) + c.rms_eps).rsqrt() * (lw.input_norm + 1)).to(torch.bfloat16)
    if kind == "linear_attention":
        assert pkg.ops.gdn_mixer_fits(x, state.conv[0], state.recurrent[0], **model._gdn_args(lw))
        general, _ = model._gdn(normed, lw, other.conv[0], other.recurrent[0])
    else:
        general = model._attention(normed, lw, other.keys[0], other.values[0], 21)
    assert metrics.compare((trace["mid"] - x).cpu(), general.float().cpu())["max_rel"] <= TOL


def _forms(tensor):
    """Other forms of a tensor: another type, shape, order in memory and alignment."""
    flat = torch.zeros((tensor.numel() + 1,), dtype=tensor.dtype, device=tensor.device)[1:].view(tensor.shape)
    strided = torch.zeros((*tensor.shape, 2), dtype=tensor.dtype, device=tensor.device)[..., 0]
    return [tensor.double(), tensor[..., :-1].contiguous(), strided, flat, tensor.cpu(), tensor.detach().requires_grad_()]


@pytest.mark.parametrize("kind", ["linear_attention", "full_attention"])
def test_the_native_mixers_take_what_the_python_form_takes(pkg, device, kind):
    """Both say which calls the kernels get: the plain one, and neither any other form of an argument."""
    c = pkg.target.small_config((kind,))
    model = pkg.target.TargetModel(pkg.target.random_weights(c, seed=9, device=device), capacity=32)
    lw, state, x = model.w.layers[0], model.synthetic_context(9, seed=4), torch.randn((4, c.hidden), device=device)
    if kind == "linear_attention":
        args = dict(hidden=x, history=state.conv[0], state=state.recurrent[0], **model._gdn_args(lw))
        plain, fits = pkg.ops.gdn_mixer_plain, pkg.ops.gdn_mixer_fits
        others = dict(key_heads=[3, 32])
    else:
        args = dict(hidden=x, keys=state.keys[0], values=state.values[0], position=9, in_proj=lw.mixer_in,
                    out_proj=lw.mixer_out, input_norm=lw.input_norm, post_norm=lw.post_norm, q_norm=lw.q_norm,
                    k_norm=lw.k_norm, inv_freq=model.inv_freq, heads=4, kv_heads=2, head_dim=128, eps=1e-6)
        plain, fits = pkg.ops.attention_mixer_plain, pkg.ops.attention_mixer_fits
        others = dict(position=[29], heads=[8], kv_heads=[1, 4], head_dim=[256, 64])
    assert plain(**args) is not None and fits(**args)
    others["in_proj"] = [args["out_proj"], args["in_proj"]._replace(packed=args["in_proj"].packed[:-32])]
    others["out_proj"] = [args["in_proj"]]
    for name, value in args.items():
        if isinstance(value, torch.Tensor):
            others[name] = _forms(value)
    for name, values in others.items():
        for value in values:
            call = {**args, name: value}
            native = plain(**call) is not None
            try:
                python = fits(**call)
            except ValueError:                          # a bank that is no bank
                python = False
            assert not native and not python, (name, getattr(value, "dtype", value), getattr(value, "shape", None))
