"""The native host path against the general one: the same calls with the native module answering None throughout
(then every argument block is filled field by field in Python), outputs and errors alike."""
import types

import pytest
import torch

from helpers import bits

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.fixture(scope="module")
def cc():
    import causal_conv1d
    return causal_conv1d


def both(cc, monkeypatch, call):
    """call() through the native module and without it: the two results, or the two exceptions as text."""
    results = []
    none = types.SimpleNamespace(**{name: (lambda *a: None) for name in
                                    ("try_fwd", "try_fwd_parts", "try_layer_block", "try_known_update", "try_update_modes",
                                     "try_decode_step", "launch_fwd", "launch_bwd")})
    for native in (cc._lib.native(), none):
        with monkeypatch.context() as m:
            m.setattr(cc._lib, "native", lambda native=native: native)
            try:
                results.append(call())
            except Exception as e:
                results.append(f"{type(e).__name__}: {e}")
    return results


def flat(r):
    return [t for x in r for t in flat(x)] if isinstance(r, (tuple, list)) else [r]


def assert_same(got, want, what):
    if isinstance(want, str) or isinstance(got, str):
        assert got == want, what
        return
    for a, b in zip(flat(got), flat(want), strict=True):
        assert a.shape == b.shape and a.stride() == b.stride() and a.dtype == b.dtype, what
        assert torch.equal(bits(a), bits(b)), what


def layouts(B, C, L, dtype, g):
    x = torch.randn(B, L, C, device=DEV, generator=g).to(dtype)
    yield "channel", x.transpose(1, 2)
    yield "time", x.transpose(1, 2).contiguous()
    yield "slice", torch.cat([x, x], -1)[..., 3:3 + C].transpose(1, 2)
    yield "batch inside", x.permute(2, 0, 1).contiguous().permute(1, 0, 2)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_prefill_and_backward(cc, monkeypatch, dtype):
    g = torch.Generator(device=DEV).manual_seed(1)
    n = 0
    for B, C, L in [(1, 24, 1), (2, 33, 77), (3, 64, 130)]:
        for name, x in layouts(B, C, L, dtype, g):
            for wtype in (dtype, torch.float32):
                W = 2 + n % 3
                w = torch.randn(C, W, device=DEV, generator=g).to(wtype)
                w = w if n % 2 else w.t().contiguous().t()
                b = None if n % 3 == 0 else torch.randn(C, device=DEV, generator=g).to(wtype if n % 4 else torch.float32)
                mask = (None if n % 2 else (torch.rand(B, L, device=DEV, generator=g) > 0.3).to(
                    [torch.int64, torch.bool, torch.float32, torch.int32, torch.uint8, torch.float16][n // 2 % 6]))
                seq = torch.arange(L, device=DEV, dtype=torch.int32).div(5, rounding_mode="floor").int().repeat(B, 1)
                init = torch.randn(B, C, 5, device=DEV, generator=g).to(dtype)
                options = dict(activation=[None, "silu", "swish"][n % 3], residual=[False, True, "masked", "unmasked", None, 2][n % 6],
                               rounding=["fused", "eager"][n % 2], attention_mask=mask)
                what = (name, B, C, L, dtype, wtype, n)
                n += 1
                assert_same(*both(cc, monkeypatch, lambda: cc.causal_conv1d_fn(x, w, b, **options)), what)
                assert_same(*both(cc, monkeypatch, lambda: cc.causal_conv1d_fn(x, w, b, seq, **options)), what)
                assert_same(*both(cc, monkeypatch, lambda: cc.causal_conv1d_fn(
                    x, w, b, initial_states=init, final_states_out=torch.zeros(B, C, 8, dtype=dtype, device=DEV), **options)), what)
                assert_same(*both(cc, monkeypatch, lambda: cc.causal_conv1d_fn(x, w, b, return_final_states=True, **options)), what)
                half = C // 2
                assert_same(*both(cc, monkeypatch, lambda: cc.causal_conv1d_fn_parts(
                    (x[:, :half], x[:, half:]), w, b, final_states_out=torch.zeros(B, C, 4, dtype=dtype, device=DEV), **options)), what)

                def train():
                    leaves = [t.detach().requires_grad_() for t in (x, w, b, init) if t is not None]
                    it = iter(leaves)
                    xx, ww, bb, ii = next(it), next(it), next(it) if b is not None else None, next(it)
                    fin = torch.zeros(B, C, 3, dtype=dtype, device=DEV)
                    y, fin = cc.causal_conv1d_fn(xx, ww, bb, initial_states=ii, final_states_out=fin, **options)
                    return torch.autograd.grad([y, fin], leaves, [torch.ones_like(y).transpose(1, 2).contiguous().transpose(1, 2),
                                                                  torch.ones_like(fin)])

                assert_same(*both(cc, monkeypatch, train), what)


def test_decode_over_pool_and_ring(cc, monkeypatch):
    g = torch.Generator(device=DEV).manual_seed(2)
    for n, (B, C, S, dtype) in enumerate([(5, 24, 4, torch.bfloat16), (3, 33, 6, torch.float32), (70, 640, 3, torch.float16)]):
        x = torch.randn(B, C, device=DEV, generator=g).to(dtype)
        w, b = torch.randn(C, 4, device=DEV, generator=g).to(dtype), torch.randn(C, device=DEV, generator=g).to(dtype)
        pool = torch.randn(B + 4, C, S, device=DEV, generator=g).to(dtype)
        idx = torch.randperm(B + 4, device=DEV, generator=g)[:B].to(torch.int32)
        idx[0] = -1
        lens = torch.randint(0, 99, (B,), device=DEV, generator=g, dtype=torch.int32)
        for options in (dict(conv_state_indices=idx), dict(cache_seqlens=lens), dict(conv_state_indices=idx, cache_seqlens=lens)):
            for mask in (None, torch.ones(B, dtype=torch.int64, device=DEV)):
                def step():
                    state = pool.clone() if "conv_state_indices" in options else pool[:B].clone()
                    y = cc.causal_conv1d_update(x, state, w, b, [None, "silu"][n % 2], token_mask=mask, residual=True, **options)
                    return y, state
                assert_same(*both(cc, monkeypatch, step), (B, C, S, dtype, list(options)))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_decode_step_of_the_layer(cc, monkeypatch, dtype):
    g = torch.Generator(device=DEV).manual_seed(3)
    for n, (B, C, S) in enumerate([(1, 640, 8), (3, 33, 4), (70, 64, 3), (2, 24, 6)]):
        wide = torch.randn(B, 3, C + 1, device=DEV, generator=g).to(dtype)
        w, b = torch.randn(C, 4, device=DEV, generator=g), torch.randn(C, device=DEV, generator=g)
        w, b = (w, b) if n == 1 else (w.to(dtype), b.to(dtype))
        start = torch.randn(B, C, S, device=DEV, generator=g).to(dtype)
        for x in (wide[:, :1, :C].contiguous(), wide[:, 1:2, 1:], wide.transpose(1, 2).contiguous().transpose(1, 2)[:, 2:, :C]):
            for mtype in (None, torch.int64, torch.bool, torch.float32):
                mask = None if mtype is None else (torch.rand(B, 9, device=DEV, generator=g) > 0.5).to(mtype)[:, ::2]

                def step():
                    state = start.clone()
                    return cc._canon_decode_step(x, state, w, b if n != 2 else None, mask, [None, "silu"][n % 2],
                                                 ["fused", "eager"][n % 2]), state
                assert_same(*both(cc, monkeypatch, step), (B, C, S, dtype, mtype))


class Tagged(torch.Tensor):
    """A subclass as a library on top of torch brings one: plain data, a type of its own."""


@pytest.mark.parametrize("layout", ["channel", "time"])
def test_tensor_subclasses_keep_their_type(cc, monkeypatch, layout):
    """empty_like of a subclass is of that subclass: outputs and input gradients are, with the native module as without."""
    g = torch.Generator(device=DEV).manual_seed(5)
    x = torch.randn(2, 40, 24, device=DEV, generator=g)
    x = x.transpose(1, 2) if layout == "channel" else x.transpose(1, 2).contiguous()
    w, b = torch.randn(24, 4, device=DEV, generator=g), torch.randn(24, device=DEV, generator=g)
    tagged = x.as_subclass(Tagged)

    def train():
        xx, ww = tagged.detach().requires_grad_(), w.detach().requires_grad_()
        y = cc.causal_conv1d_fn(xx, ww, b, activation="silu", residual=True)
        return y.detach(), torch.autograd.grad(y.as_subclass(torch.Tensor).sum(), [xx, ww])

    for call in (lambda: cc.causal_conv1d_fn(tagged, w, b), train, lambda: cc._launch_fwd(tagged, w, b, None, None, None, 0, 0, 0),
                 lambda: cc.causal_conv1d_fn_parts([tagged[:, :8], tagged[:, 8:]], w, b),
                 lambda: cc._launch_bwd(tagged, tagged, w, b, None, torch.empty(24, 4, device=DEV), torch.empty(24, device=DEV), 0, 0)):
        native, general = both(cc, monkeypatch, call)
        assert_same(native, general, layout)
        assert [type(t) for t in flat(native)] == [type(t) for t in flat(general)]
        assert type(flat(native)[0]) is Tagged


def test_refused_calls(cc, monkeypatch):
    x, w, b = torch.randn(2, 8, 16, device=DEV), torch.randn(8, 4, device=DEV), torch.randn(8, device=DEV)
    mask, pool = torch.ones(2, 16, device=DEV), torch.randn(4, 8, 4, device=DEV)
    idx = torch.zeros(2, dtype=torch.int32, device=DEV)
    fn, parts, update = cc.causal_conv1d_fn, cc.causal_conv1d_fn_parts, cc.causal_conv1d_update
    calls = [lambda: fn(x[0], w), lambda: fn(x.double(), w), lambda: fn(x, w[:7]), lambda: fn(x, torch.randn(8, 5, device=DEV)),
             lambda: fn(x, w.cpu()), lambda: fn(x, w, b[:7]), lambda: fn(x, w, b.cpu()), lambda: fn(x, w, b, activation="relu"),
             lambda: fn(x, w, b, residual="other"), lambda: fn(x, w, b, rounding="other"), lambda: fn(x, w, b, attention_mask=mask[:1]),
             lambda: fn(x, w, b, attention_mask=mask.double()), lambda: fn(x, w, b, attention_mask=mask.cpu()),
             lambda: fn(x, w, b, idx), lambda: fn(x, w, b, torch.zeros(2, 16, device=DEV)),
             lambda: fn(x, w, b, torch.zeros(2, 16, dtype=torch.int32, device=DEV), initial_states=x[..., :4]),
             lambda: fn(x, w, b, initial_states=x[..., :2]), lambda: fn(x, w, b, initial_states=x[:1, :, :4]),
             lambda: fn(x, w, b, final_states_out=x[:, :, :0]), lambda: fn(x, w, b, final_states_out=x.half()),
             lambda: fn(x, w, b, final_states_out=torch.zeros(2, 8, 65, device=DEV)), lambda: fn(x[..., :0], w, b),
             lambda: parts([x, x[:, :, :8]], w), lambda: parts([x] * 5, w), lambda: parts([x, x.half()], w), lambda: parts([x[:, :4]], w),
             lambda: update(x[..., 0], pool, w, b, conv_state_indices=idx.long()), lambda: update(x[..., 0], pool, w, b, cache_seqlens=idx),
             lambda: update(x[..., 0], pool[:, :7], w, b, conv_state_indices=idx), lambda: update(x[..., 0], pool[..., :2], w, b, conv_state_indices=idx),
             lambda: update(x[..., 0], pool.half(), w, b, conv_state_indices=idx), lambda: update(x[..., 0], pool, w, b, conv_state_indices=idx[:1])]
    for n, call in enumerate(calls):
        native, general = both(cc, monkeypatch, call)
        assert_same(native, general, n)


def test_decode_call_of_the_wrong_rank(cc, monkeypatch):
    """A bias or a token mask of another rank than one is refused before its sizes enter the call's signature, whose length
    is that of the ranks that are taken (a bias and a mask of three dimensions each would not fit it)."""
    x, w, b = torch.randn(2, 8, device=DEV), torch.randn(8, 4, device=DEV), torch.randn(8, device=DEV)
    state, mask = torch.randn(2, 8, 3, device=DEV), torch.ones(2, device=DEV)
    for bias in (b, b[None, :], b[None, :, None], b[0]):
        for m in (None, mask, mask[:, None], mask[:, None, None], mask[0]):
            native, general = both(cc, monkeypatch, lambda: cc.causal_conv1d_update(x, state.clone(), w, bias, token_mask=m))
            assert_same(native, general, (bias.shape, None if m is None else m.shape))
            assert isinstance(native, str) == (bias.dim() != 1 or (m is not None and m.dim() != 1))
            if bias.dim() != 1:
                assert native == f"ValueError: Expected 1D bias tensor, got {bias.dim()}D"


def test_decode_signatures_without_the_native_module(cc, monkeypatch):
    """Where the native module declines (another device than the current one, a module built for another torch) a decode call
    that was checked once is launched from its argument block as well, and no other call is."""
    x, w, b = torch.randn(2, 8, device=DEV), torch.randn(8, 4, device=DEV), torch.randn(8, device=DEV)
    state, mask = torch.randn(2, 8, 4, device=DEV), torch.tensor([1.0, 0.5], device=DEV)
    calls = [lambda s: cc.causal_conv1d_update(x, s, w), lambda s: cc.causal_conv1d_update(x, s, w, b, "silu", token_mask=mask, residual=True),
             lambda s: cc.causal_conv1d_update(x.t().contiguous().t(), s, w, b, rounding="eager")]
    monkeypatch.setattr(cc._update_tls, "known", {}, raising=False)
    states = [[state.clone() for _ in calls] for _ in range(2)]
    want = [[call(s) for call, s in zip(calls, row)] for row in states for _ in range(2)]
    assert len(cc._known_updates()) == len(calls) and all(type(key) is bytes for key in cc._known_updates())   # (the module's own)
    monkeypatch.setattr(cc._update_tls, "known", {})
    monkeypatch.setattr(cc._lib, "native", cc._lib._OtherTorch)
    launch, checked = cc._launch_update, []
    monkeypatch.setattr(cc, "_launch_update", lambda *a: checked.append(1) or launch(*a))
    again = [[state.clone() for _ in calls] for _ in range(2)]
    got = [[call(s) for call, s in zip(calls, row)] for row in again for _ in range(2)]
    assert_same(got, want, "outputs")
    assert_same(again, states, "states")
    assert len(checked) == len(calls) == len(cc._known_updates())
    calls[0](state.half().float()[:, :, 1:])                                   # another stride of the state
    cc.causal_conv1d_update(x[..., None], state, w)                            # another rank of x
    with torch.enable_grad():
        cc.causal_conv1d_update(x, state.clone(), w.clone().requires_grad_())  # gradients
    assert len(checked) == len(calls) + 3
    for bad in (lambda: cc.causal_conv1d_update(x, state, w, activation=["relu"]), lambda: cc.causal_conv1d_update(x, state, w[:7])):
        with pytest.raises((ValueError, NotImplementedError)):
            bad()


def test_another_stream_and_a_captured_graph(cc):
    x = torch.randn(2, 64, 256, device=DEV).bfloat16()
    w = torch.randn(64, 4, device=DEV).bfloat16()
    want = cc.causal_conv1d_fn(x, w)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        got = cc.causal_conv1d_fn(x, w)
    side.synchronize()
    assert torch.equal(bits(got), bits(want))
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = cc.causal_conv1d_fn(x, w)
    for i in range(3):
        x.copy_(torch.randn(2, 64, 256, device=DEV).bfloat16())
        want = cc.causal_conv1d_fn(x, w)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(bits(out), bits(want)), i


@pytest.mark.parametrize("layout", ["channel", "time"])
def test_training_call(cc, monkeypatch, layout):
    """The native autograd node against the Python one: gradients of every subset of the inputs, a gradient of the output in
    another layout or expanded, a graph walked twice, saved-tensor hooks; and what is refused stays refused with the same
    words (a saved input written to, a graph walked a second time, transforms, forward mode, double backward)."""
    g = torch.Generator(device=DEV).manual_seed(4)
    B, C, L = 2, 24, 70
    x0 = torch.randn(B, L, C, device=DEV, generator=g).bfloat16()
    x0 = x0.transpose(1, 2) if layout == "channel" else x0.transpose(1, 2).contiguous()
    d0 = torch.randn(B, C, L, device=DEV, generator=g).bfloat16()
    m = torch.ones(B, L, dtype=torch.int64, device=DEV)
    m[1, 50:] = 0
    seq = torch.arange(L, device=DEV, dtype=torch.int32).div(9, rounding_mode="floor").int().repeat(B, 1)
    for wtype in (torch.bfloat16, torch.float32):
        w0, b0 = torch.randn(C, 4, device=DEV, generator=g).to(wtype), torch.randn(C, device=DEV, generator=g).to(wtype)

        def leaves(which=(1, 1, 1)):
            return [t.detach().clone(memory_format=torch.preserve_format).requires_grad_(bool(r)) for t, r in zip((x0, w0, b0), which)]

        for which in ((1, 1, 1), (1, 0, 0), (0, 1, 0), (0, 0, 1), (0, 1, 1)):
            for options in (dict(), dict(attention_mask=m, activation="silu", residual=True), dict(seq_idx=seq, residual="unmasked")):
                def grads(d=d0):
                    t = leaves(which)
                    y = cc.causal_conv1d_fn(*t, **options)
                    return (y.detach(), *torch.autograd.grad(y, [v for v in t if v.requires_grad], d))
                assert_same(*both(cc, monkeypatch, grads), (which, list(options)))
        for d in (d0.transpose(1, 2).contiguous().transpose(1, 2), d0[:1, :1, :1].expand(B, C, L)):
            assert_same(*both(cc, monkeypatch, lambda: grads(d)), "dout")

        def twice():
            x, w, b = leaves()
            y = cc.causal_conv1d_fn(x, w, b, activation="silu")
            first = torch.autograd.grad(y, (x, w, b), d0, retain_graph=True)
            return first, torch.autograd.grad(y, (x, w, b), d0)
        assert_same(*both(cc, monkeypatch, twice), "twice")

        packed = []

        def hooked():
            packed.clear()
            x, w, b = leaves()
            with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(1) or t.cpu(), lambda t: t.to(DEV)):
                y = cc.causal_conv1d_fn(x, w, b, attention_mask=m)
            return torch.autograd.grad(y, (w, b), d0), len(packed)
        (got, n), (want, n_want) = both(cc, monkeypatch, hooked)
        assert_same(got, want, "hooks")
        assert n == n_want == 4

        def written():
            x, w, b = leaves()
            y = cc.causal_conv1d_fn(x, w, b)
            with torch.no_grad():
                w.add_(1)
            return torch.autograd.grad(y, (x, w, b), d0)

        def freed():
            x, w, b = leaves()
            y = cc.causal_conv1d_fn(x, w, b)
            torch.autograd.grad(y, (x, w, b), d0)
            return torch.autograd.grad(y, (x, w, b), d0)

        def transform():
            x, w, b = leaves((0, 0, 0))
            return torch.func.grad(lambda v: cc.causal_conv1d_fn(v, w, b).float().sum())(x)

        def mapped():
            x, w, b = leaves((0, 1, 1))
            return torch.func.vmap(lambda v: cc.causal_conv1d_fn(v, w, b))(torch.stack([x, x]))

        def forward_mode():
            x, w, b = leaves()
            with torch.autograd.forward_ad.dual_level():
                dual = torch.autograd.forward_ad.make_dual(x, torch.ones_like(x))
                return cc.causal_conv1d_fn(dual, w, b).sum()

        def second():
            x, w, b = leaves()
            y = cc.causal_conv1d_fn(x, w, b, activation="silu")
            gx, = torch.autograd.grad(y, x, d0, create_graph=True)
            return torch.autograd.grad(gx.float().sum(), x)
        for call, words in ((written, "modified by an inplace operation"), (freed, "backward through the graph a second time"),
                            (transform, "functorch transforms"), (mapped, "functorch transforms"), (forward_mode, "forward mode AD"),
                            (second, "its gradients cannot be differentiated")):
            got, want = both(cc, monkeypatch, call)
            assert got == want and words in got, (call.__name__, got, want)


@pytest.mark.parametrize("activation", [None, "silu"])
def test_a_graph_of_the_backward(cc, monkeypatch, activation):
    """create_graph=True: the gradients themselves are as without, and a loss that differentiates one of them again is refused,
    also where another term of it has a gradient of its own; one that does not depend on the variable asked for is not."""
    g = torch.Generator(device=DEV).manual_seed(6)
    B, C, L, S = 2, 24, 40, 4
    x0, t0 = torch.randn(B, C, L, device=DEV, generator=g), torch.randn(B, C, device=DEV, generator=g)
    w0, b0 = torch.randn(C, 4, device=DEV, generator=g), torch.randn(C, device=DEV, generator=g)
    s0 = torch.randn(B, C, S, device=DEV, generator=g)

    def fn(x, w, b, s):
        return [cc.causal_conv1d_fn(x, w, b, activation=activation)]

    def packed(x, w, b, s):
        return [cc.causal_conv1d_fn(x, w, b, torch.zeros(B, L, dtype=torch.int32, device=DEV), activation=activation)]

    def states(x, w, b, s):
        return cc.causal_conv1d_fn(x, w, b, initial_states=s, final_states_out=torch.empty(B, C, S, device=DEV), activation=activation)

    def parts(x, w, b, s):
        ys, fin = cc.causal_conv1d_fn_parts(x.split([8, 16], 1), w, b, initial_states=s, activation=activation,
                                            final_states_out=torch.empty(B, C, S, device=DEV))
        return [*ys, fin]

    def update(x, w, b, s):
        s = s * 1
        return [cc.causal_conv1d_update(x[..., 0], s, w, b, activation), s]

    def update_parts(x, w, b, s):
        s = s * 1
        return [*cc.causal_conv1d_update_parts(x[..., 0].split([8, 16], 1), s, w, b, activation), s]

    for call in (fn, packed, states, parts, update, update_parts):
        n = 3 if call in (fn, packed) else 4

        def leaves():
            return [t.clone().requires_grad_() for t in (x0, w0, b0, s0)]

        def first(create_graph):
            t = leaves()
            loss = sum(y.square().sum() for y in call(*t))
            return torch.autograd.grad(loss, t[:n], create_graph=create_graph)
        for plain, again in zip(both(cc, monkeypatch, lambda: first(False)), both(cc, monkeypatch, lambda: first(True))):
            assert_same([v.detach() for v in again], list(plain), call.__name__)

        # the gradient of a linear loss in variable i, squared, beside a term of its own: its derivative in variable j
        for i in range(n):
            for j in range(n):
                def mixed(second=True):
                    t = leaves()
                    y = call(*t)
                    gi, = torch.autograd.grad(sum(v.sum() for v in y), t[i], create_graph=True)
                    loss = sum(v.square().sum() for v in t) + (gi.square().sum() if second else 0)
                    return torch.autograd.grad(loss, t[j])
                # without an activation y is bilinear: dx and the state's gradient depend on the taps, the taps' on x and state
                depends = activation is not None or (i in (0, 3) and j == 1) or (i == 1 and j in (0, 3))
                for got in both(cc, monkeypatch, mixed):
                    if depends:
                        assert isinstance(got, str) and "its gradients cannot be differentiated" in got, (call.__name__, i, j, got)
                    else:
                        assert_same(got, mixed(second=False), (call.__name__, i, j))


def test_blocks_of_the_layer(cc, monkeypatch):
    """CanonLayer's block call: one tensor and parts, with and without a cache, a continued state, masks, x that is not
    dense; outputs, their strides and the cached states as through the functions."""
    from causal_conv1d.canon import CanonLayer
    g = torch.Generator(device=DEV).manual_seed(5)
    for n, dtype in enumerate([torch.bfloat16, torch.float32, torch.float16]):
        dims, B, T = ((16, 8, 8), (12, 12), (33,))[n], 3, 21
        C = sum(dims)
        config = types.SimpleNamespace(canon_kernel=4, canon_bias=n != 1, canon_activation=n == 0)
        layer = CanonLayer(C, config, "b", rounding=("fused", "eager")[n == 2]).to(DEV, dtype).requires_grad_(False)
        x = torch.randn(B, T, C, device=DEV, generator=g).to(dtype)
        forms = [x, x.transpose(1, 2).contiguous().transpose(1, 2), torch.cat([x, x], -1)[..., 1:1 + C], x[:, :2]]
        for xs in forms:
            mask = torch.ones(B, xs.shape[1] + 5, dtype=torch.int64, device=DEV)
            mask[1, -3:] = 0
            for m in (None, mask, mask[:, 5:]):
                def one():
                    cache = types.SimpleNamespace(_max_layers=2)
                    y = layer(xs, m), layer(xs, m, cache, 1), layer(xs, m, cache, 1)
                    return y, cache.canon_cache_b[1]

                def parts():
                    cache = types.SimpleNamespace(_max_layers=2)
                    p = xs.split(dims, -1)
                    y = layer.forward_parts(p, m), layer.forward_parts(list(p), m, cache, 0), layer.forward_parts(p, m, cache, 0)
                    return y, cache.canon_cache_b[0]
                for call in (one, parts):
                    assert_same(*both(cc, monkeypatch, call), (dtype, xs.stride(), call.__name__))
