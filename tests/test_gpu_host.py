"""GPU: the native form of ops.py's plain calls (``csrc/host.cpp``) against the Python form of the same calls.

Both enqueue the same kernels with the same arguments, so results are equal bit for bit; what the native form does not
take (views, other types, subclasses, modes) it leaves to the Python form, errors included.
"""
import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

pytestmark = pytest.mark.gpu


@pytest.fixture
def python_form(pkg, monkeypatch):
    """Calls a function with the native form switched off."""
    def call(fn, *args, **kw):
        with monkeypatch.context() as m:
            m.setattr(pkg.ops, "_plain", lambda x: False)
            return fn(*args, **kw)
    return call


def _weight(pkg, device, n, k, group=128, dtype=torch.bfloat16, layout="tiled", seed=0):
    w = pkg.synthetic.int4_weight(torch.Generator().manual_seed(seed), (n, k), group, dtype).to(device)
    return w.tiled() if layout == "tiled" else w


@pytest.mark.parametrize("shape", [(2048,), (1, 2048), (2, 3, 2048), (70, 2048)])
@pytest.mark.parametrize("group,dtype,layout", [(128, torch.bfloat16, "tiled"), (256, torch.float32, "portable")])
def test_linear(pkg, device, python_form, shape, group, dtype, layout):
    w = _weight(pkg, device, 96, 2048, group, dtype, layout)
    x = torch.randn(shape, device=device).to(torch.bfloat16)
    for out_dtype in (torch.bfloat16, torch.float32):
        y = pkg._lib.host().linear(x, w, out_dtype is torch.float32)
        want = python_form(pkg.ops.qlinear, x, w, out_dtype=out_dtype)
        assert y is not None and y.dtype == out_dtype and y.shape == (*shape[:-1], 96) and torch.equal(y, want)


def test_linear_leaves_other_forms(pkg, device, python_form):
    w, x = _weight(pkg, device, 96, 512), torch.randn((8, 512), device=device).to(torch.bfloat16)
    native = pkg._lib.host().linear
    strided = torch.randn((8, 1024), device=device).to(torch.bfloat16)[:, ::2]
    assert native(strided, w, False) is None
    assert torch.equal(pkg.ops.qlinear(strided, w), pkg.ops.qlinear(strided.contiguous(), w))
    offset = torch.randn((8 * 512 + 1,), device=device).to(torch.bfloat16)[1:].view(8, 512)      # 2-byte aligned
    for bad, error in ((offset, pkg._lib.DflashError), (x.float(), ValueError), (x[:, :256], ValueError), (x.cpu(), ValueError)):
        with pytest.raises(error):
            pkg.ops.qlinear(bad, w)
    assert pkg.ops.qlinear(x[:0], w).shape == (0, 96)
    for bad in (w._replace(group_size=64), w._replace(layout="other"), w._replace(scales=w.scales.half()),
                w._replace(scales=w.scales[:, :1]), w._replace(packed=w.packed.cpu())):
        assert native(x, bad, False) is None
        with pytest.raises(ValueError):
            pkg.ops.qlinear(x, bad)
    assert native(x, tuple(w), False) is None

    class Mode(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))
    with Mode():
        assert native(x, w, False) is None
        assert pkg.ops.qlinear(x, w).shape == (8, 96)


@pytest.mark.parametrize("tokens,shared", [(1, True), (16, False), (40, True)])
def test_moe(pkg, device, python_form, tokens, shared):
    layer = pkg.synthetic.moe_layer(tokens, hidden=512, inter=512, experts=16, seed=tokens)
    x, banks = layer.hidden.to(device), (layer.gate_up.to(device), layer.down.to(device))
    sh = pkg.SharedExpert(layer.shared.gate_up.to(device), layer.shared.down.to(device), layer.shared.gate_weight.to(device))
    router, native = layer.router_weight.to(device), pkg._lib.host().moe
    args = dict(top_k=4, router_weight=router, shared=sh if shared else None)
    want = python_form(pkg.ops.moe_w4a16, x, *banks, **args)
    need = pkg.ops.moe_workspace_bytes(tokens, 512, 512, 16, 4, 128, shared)
    for ws in (None, torch.empty(need, dtype=torch.uint8, device=device)):
        got = native(x, *banks, 4, router, args["shared"], ws, None)
        assert got is not None and torch.equal(got, want)
    assert native(x, *banks, 4, router, args["shared"], torch.empty(need - 1, dtype=torch.uint8, device=device), None) is None
    assert native(x, *banks, 4, router.t().contiguous().t(), args["shared"], None, None) is None
    for k in (0, 17, True, 4.0):
        assert native(x, *banks, k, router, args["shared"], None, None) is None


@pytest.mark.parametrize("kind", ["linear_attention", "full_attention"])
@pytest.mark.parametrize("tokens", [1, 16, 30])
def test_layer(pkg, device, python_form, kind, tokens):
    c = pkg.target.small_config((kind,))
    model = pkg.target.TargetModel(pkg.target.random_weights(c, seed=3, device=device, layout="tiled"), capacity=80)
    x = torch.randn((tokens, c.hidden), device=device)

    def run():
        state = model.synthetic_context(9, seed=4)
        hidden, pending = model.layer(0, x, state)
        model.commit(state, pkg.target.Pending(9, tokens, [pending]), max(1, tokens - 3))
        return [hidden, *state.conv, *state.recurrent, *state.keys, *state.values]
    for a, b in zip(run(), python_form(run)):
        assert (a is None and b is None) or torch.equal(a, b)


def test_calls_run_on_the_current_stream(pkg, device):
    """A call inside a stream context is ordered on that stream: behind work queued there, before what follows."""
    w, stream = _weight(pkg, device, 512, 2048), torch.cuda.Stream(device)
    x = torch.randn((16, 2048), device=device).to(torch.bfloat16)
    want = pkg.ops.qlinear(x, w)
    torch.cuda.synchronize()
    late = torch.zeros_like(x)
    with torch.cuda.stream(stream):
        big = torch.randn((4096, 4096), device=device)
        for _ in range(8):
            big = big @ big
            big /= big.norm()
        late.copy_(x)
        y = pkg.ops.qlinear(late, w)
    stream.synchronize()
    assert torch.equal(y, want)


@pytest.mark.parametrize("tokens,hidden", [(1, 512), (3, 2048), (70, 8192)])
def test_rms_norm(pkg, device, tokens, hidden):
    """The one-launch final norm against the norm in 64 bits: a few fp32 roundings (2^-24 each)."""
    x = torch.randn((tokens, hidden), device=device) * 3
    w = torch.randn((hidden,), device=device)
    y = pkg.ops.rms_norm(x, w, 1e-6)
    want = x.double() * (x.double().square().mean(-1, keepdim=True) + 1e-6).rsqrt() * (w.double() + 1)
    assert ((y - want).norm() / want.norm()).item() <= 3e-7
    assert pkg.ops.rms_norm(x.to(torch.bfloat16), w, 1e-6) is None
    assert pkg.ops.rms_norm(x[:, ::2], w[::2], 1e-6) is None
    assert pkg.ops.rms_norm(x.requires_grad_(), w, 1e-6) is None


@pytest.mark.parametrize("tokens", [1, 2, 15, 16, 17, 18, 19, 35])
def test_commit_of_a_whole_block_takes_the_windows_tail(pkg, device, tokens):
    """The conv history after a whole block, also where the last chunk holds fewer tokens than the taps."""
    c = pkg.target.small_config(("linear_attention",))
    layout = "tiled" if tokens <= 32 else "portable"
    model = pkg.target.TargetModel(pkg.target.random_weights(c, seed=3, device=device, layout=layout), capacity=80)
    state = model.synthetic_context(9, seed=4)
    _, pending = model.layer(0, torch.randn((tokens, c.hidden), device=device), state)
    model.commit(state, pkg.target.Pending(9, tokens, [pending]), tokens)
    assert torch.equal(state.conv[0], pending.window[:, :, tokens:])
    assert state.conv[0].untyped_storage().nbytes() == state.conv[0].nbytes


def test_calls_without_the_native_form(pkg, device, monkeypatch):
    """Where dflash_host.so cannot be loaded the Python form serves every call, with the same bits."""
    w, x = _weight(pkg, device, 96, 512), torch.randn((8, 512), device=device).to(torch.bfloat16)
    c = pkg.target.small_config()
    model = pkg.target.TargetModel(pkg.target.random_weights(c, seed=3, device=device), capacity=80)
    ids = torch.arange(8, device=device)

    def run():
        state = model.synthetic_context(9, seed=4)
        out = model.forward(ids, state)
        model.commit(state, out.pending, 5)
        return [pkg.ops.qlinear(x, w), out.top1, *(r for r in state.recurrent if r is not None)]
    want = run()
    monkeypatch.setattr(pkg._lib, "_HOST", False)
    assert pkg._lib.host() is None
    for a, b in zip(run(), want):
        assert torch.equal(a, b)


@pytest.mark.parametrize("tokens,accepted", [(1, 1), (9, 9), (16, 16), (17, 17), (32, 32), (16, 5), (32, 16)])
def test_two_commits_of_one_block_share_nothing(pkg, device, tokens, accepted):
    """States committed from one pending record have tensors of their own: writing one in place changes neither the
    others, also of commits that follow, nor the state before the block."""
    c = pkg.target.small_config(("linear_attention",))
    model = pkg.target.TargetModel(pkg.target.random_weights(c, seed=3, device=device), capacity=80)
    state = model.synthetic_context(9, seed=4)
    before = state.clone()
    x = torch.randn((tokens, c.hidden), generator=torch.Generator().manual_seed(tokens)).to(device)
    _, pending = model.layer(0, x, state)
    # states rebuilt from the record differ by fp32 sums in another order and by decays e^(G_j - G_s) of log decays held
    # in fp32, each 2^-24 |G| off
    bound = 1e-6 + 2.0 ** -23 * pending.chunks[-1].cum.abs().max().item()
    conv, chunks = pending.window[:, :, accepted:accepted + 3].clone(), pending.chunks
    want = pkg.layers.state_after(chunks[-2].state if len(chunks) > 1 else state.recurrent[0], chunks[-1].keys, chunks[-1].u,
                                  chunks[-1].cum, accepted - 16 * (len(chunks) - 1)) if accepted == tokens else None
    commits = []
    for _ in range(3):
        branch = pkg.target.TargetState(9, list(state.conv), list(state.recurrent), state.keys, state.values)
        model.commit(branch, pkg.target.Pending(9, tokens, [pending]), accepted)
        want = branch.recurrent[0].clone() if want is None else want
        assert torch.equal(branch.conv[0], conv)
        assert ((branch.recurrent[0] - want).norm() / want.norm()).item() <= bound
        branch.conv[0].fill_(1)
        branch.recurrent[0].fill_(1)
        commits.append(branch)
    assert len({t.untyped_storage().data_ptr() for b in commits for t in (b.conv[0], b.recurrent[0])}) == 6
    assert torch.equal(state.conv[0], before.conv[0]) and torch.equal(state.recurrent[0], before.recurrent[0])


def test_rms_norm_of_more_rows_than_one_launch_holds(pkg, device):
    """2^23 + 3 rows at 512 threads each are more than 2^32 work-items: three launches (4 columns, in place)."""
    tokens = (1 << 23) + 3
    x = torch.randn((tokens, 4), device=device)
    w = torch.randn((4,), device=device)
    want = x * (x.square().mean(-1, keepdim=True) + 1e-6).rsqrt() * (w + 1)
    pkg._lib.call("dflash_rms_norm", pkg.ops._ptr(x), tokens, 4, pkg.ops._ptr(w), 1e-6, pkg.ops._ptr(x), pkg.ops._stream(device))
    torch.testing.assert_close(x, want, rtol=1e-6, atol=1e-6)     # a few fp32 roundings each
