"""Module-level parity on the GPU: the reference's GPU tests re-stated for the native path
(tests/test_lookahead.py:67-143, 185-222, 225-282 of the reference) and the benchmark configurations at
their full sizes, checked through the oracle on sampled heads and through size-independent
properties (parallel == cached sequential, causality / prefix invariance)."""
import pytest
import torch

pytestmark = pytest.mark.gpu

from oracle import castle_oracle as O

DEV = "cuda:0"


def make(dim, heads, d, dtype=torch.float32, prenorm=False, rotary=False, seed=0):
    from lookahead_keys_attention_amd import Castle

    torch.manual_seed(seed)
    m = Castle(dim, heads=heads, dim_head=d, use_triton=True, prenorm=prenorm, rotary_emb=rotary)
    return m.to(DEV).to(dtype)


def cpu_params(m):
    return {k: v.detach().cpu().float() for k, v in m.state_dict().items()}


def bf16_close(got, ref, what):
    got, ref = got.detach().cpu().double(), ref.detach().cpu().double()
    err = (got - ref).abs().max().item()
    rel = ((got - ref).norm() / ref.norm()).item()
    assert err <= 2e-2 * ref.abs().max().item() and rel <= 2e-2, f"{what}: max err {err:.3e} (max {ref.abs().max():.3e}), rel {rel:.3e}"


@pytest.mark.parametrize("prenorm", [False, True])
def test_native_vs_oracle_forward_and_grads(prenorm):
    # reference: test_castle_triton_vs_reference, B2 L256 dim128 d64 H2, fwd 1e-3, grads 2e-2
    m = make(128, 2, 64, prenorm=prenorm)
    p = {k: v.clone().requires_grad_() for k, v in cpu_params(m).items()}
    x = torch.randn(2, 256, 128, generator=torch.Generator().manual_seed(1))
    gy = torch.randn(2, 256, 128, generator=torch.Generator().manual_seed(2))
    xg = x.to(DEV).requires_grad_()
    y = m(xg)
    y.backward(gy.to(DEV))
    xr = x.clone().requires_grad_()
    yr = O.module_forward(xr, p, 2)
    yr.backward(gy)
    assert (y.detach().cpu() - yr.detach()).abs().max() <= 1e-3
    assert (xg.grad.cpu() - xr.grad).abs().max() <= 2e-2
    for name, par in m.named_parameters():
        assert (par.grad.cpu() - p[name].grad).abs().max() <= 2e-2, name


@pytest.mark.parametrize("prenorm", [False, True])
def test_native_causality(prenorm):
    # reference: test_castle_causality_triton, B2 L64 dim128 d64 H2, atol 1e-3
    m = make(128, 2, 64, prenorm=prenorm).eval()
    x = torch.randn(2, 64, 128, generator=torch.Generator().manual_seed(3)).to(DEV)
    with torch.no_grad():
        assert (m(x)[:, :32] - m(x[:, :32])).abs().max() <= 1e-3


@pytest.mark.parametrize("prenorm", [False, True])
@pytest.mark.parametrize("rotary", [False, True])
def test_native_parallel_vs_sequential(prenorm, rotary):
    # reference: test_castle_triton_parallel_vs_sequential, B2 L16 dim32 d16 H2 split 8, atol 1e-3.
    # Here the cached steps run in HIP as well, and the rotary variant is included.
    from lookahead_keys_attention_amd import Cache

    m = make(32, 2, 16, prenorm=prenorm, rotary=rotary).eval()
    x = torch.randn(2, 16, 32, generator=torch.Generator().manual_seed(4)).to(DEV)
    with torch.no_grad():
        y0, cache = m(x[:, :8], return_next_cache=True)
        ys = [y0]
        for t in range(8, 16):
            y, cache = m(x[:, t:t + 1], cache=cache, return_next_cache=True)
            ys.append(y)
        full = m(x)
    assert isinstance(cache, Cache) and cache.U.shape == (2, 2, 16, 16)
    assert (torch.cat(ys, 1) - full).abs().max() <= 1e-3


def test_decode_from_scratch_and_from_plain_tuple():
    m = make(64, 2, 32).eval()
    p = cpu_params(m)
    x = torch.randn(2, 6, 64, generator=torch.Generator().manual_seed(5))
    with torch.no_grad():
        cache, ys = None, []
        for t in range(6):
            y, cache = m(x[:, t:t + 1].to(DEV), cache=cache)
            ys.append(y)
        ref = O.module_forward(x, p, 2)
        assert (torch.cat(ys, 1).cpu() - ref).abs().max() <= 1e-3
        # a foreign 4-tuple (e.g. produced by the dense formulation) is copied, then advanced
        _, oc = O.module_forward(x[:, :5], p, 2, return_next_cache=True)
        y5, c5 = m(x[:, 5:].to(DEV), cache=tuple(t.to(DEV) for t in oc))
        assert (y5.cpu() - ref[:, 5:]).abs().max() <= 1e-3 and c5.U.shape[-2] == 6
        # an already-advanced native cache cannot be replayed
        _, c_old = m(x[:, :3].to(DEV), return_next_cache=True)
        m(x[:, 3:4].to(DEV), cache=c_old)
        with pytest.raises(RuntimeError, match="in place"):
            m(x[:, 3:4].to(DEV), cache=c_old)


def test_reading_the_lookahead_keys_mid_window_completes_them():
    """The native step writes U back on every 4th step only.  Whoever reads `cache.U` in between gets
    the pending tokens folded in first (so the tensor seen is always the true U), and the steps that
    follow carry on from there: outputs and keys equal the oracle's, whether U was read or not."""
    m = make(64, 2, 32).eval()
    p = cpu_params(m)
    x = torch.randn(2, 14, 64, generator=torch.Generator().manual_seed(6))
    ref = O.module_forward(x, p, 2)
    for read_at in ((), (6, 7, 9), (5,)):
        with torch.no_grad():
            _, cache = m(x[:, :3].to(DEV), return_next_cache=True)
            ys = []
            for t in range(3, 14):
                y, cache = m(x[:, t:t + 1].to(DEV), cache=cache)
                ys.append(y)
                if t in read_at:
                    _, oc = O.module_forward(x[:, :t + 1], p, 2, return_next_cache=True)
                    assert (cache.U.cpu() - oc.U).abs().max() <= 1e-3, f"U read after step {t}"
                    assert cache._store.pending() == 0
            assert (torch.cat(ys, 1).cpu() - ref[:, 3:]).abs().max() <= 1e-3
            _, oc = O.module_forward(x, p, 2, return_next_cache=True)
            U, qu_c, kc_c, vc_c = cache            # unpacking reads U too
            assert (U.cpu() - oc.U).abs().max() <= 1e-3 and (kc_c.cpu() - oc.kc_cache).abs().max() <= 1e-5


def test_single_token_step_with_grad_mode_on():
    """The native cached step is inference-only.  Castle(use_triton=True) says so when a single-token
    call would need a graph (grad mode on, parameters requiring grad) instead of silently going
    dense; an auto-selected module (use_triton=None) takes the differentiable dense step, as the
    reference's module would, and warns once that the native cache is copied out."""
    from lookahead_keys_attention_amd import Castle

    m = make(32, 2, 16)
    x = torch.randn(1, 6, 32).to(DEV)
    with torch.no_grad():
        _, cache = m(x[:, :5], return_next_cache=True)
    with pytest.raises(RuntimeError, match="inference-only"):
        m(x[:, 5:], cache=cache)
    with torch.no_grad():
        want, _ = m(x[:, 5:], cache=cache)
    torch.manual_seed(0)
    auto = Castle(32, heads=2, dim_head=16, use_triton=None).to(DEV)
    auto.load_state_dict(m.state_dict())
    with torch.no_grad():
        _, cache = auto(x[:, :5], return_next_cache=True)
    Castle._warned_dense_step = False
    with pytest.warns(RuntimeWarning, match="dense PyTorch step"):
        got, nxt = auto(x[:, 5:], cache=cache)
    assert got.requires_grad and nxt.U.shape[-2] == 6
    got.sum().backward()
    assert auto.to_all_qkv.weight.grad is not None
    assert (got.detach() - want).abs().max() <= 1e-4


def test_projection_over_many_rows_forms_its_weight_gradient_in_row_ranges():
    """castle._linear: above SPLIT_WGRAD_MIN_ROWS rows the weight gradient of a bias-free projection is
    summed from partial products over row ranges; output and both gradients equal nn.Linear's (the
    partial products are kept in fp32, so the one rounding at the end is the same)."""
    from lookahead_keys_attention_amd import castle as C

    torch.manual_seed(5)
    layer = torch.nn.Linear(96, 160, bias=False).to(DEV).bfloat16()
    x = torch.randn(4, C.SPLIT_WGRAD_MIN_ROWS // 4, 96, device=DEV).bfloat16().requires_grad_()
    gy = torch.randn(4, C.SPLIT_WGRAD_MIN_ROWS // 4, 160, device=DEV).bfloat16()
    y = C._linear(layer, x)
    assert y.grad_fn is not None and "ManyRowLinear" in type(y.grad_fn).__name__
    y.backward(gy)
    got = (y.detach(), x.grad.clone(), layer.weight.grad.clone())
    x.grad, layer.weight.grad = None, None
    y2 = layer(x)
    y2.backward(gy)
    assert torch.equal(got[0], y2.detach()) and torch.equal(got[1], x.grad)
    ref = gy.float().flatten(0, 1).t() @ x.detach().float().flatten(0, 1)
    bf16_close(got[2], ref, "weight gradient in row ranges")
    assert (got[2].float() - ref).norm() <= 1.05 * (layer.weight.grad.float() - ref).norm()
    # few rows, no grad mode, fp32: the layer itself
    small = C._linear(layer, x[:, :8])
    assert "ManyRowLinear" not in type(small.grad_fn).__name__
    with torch.no_grad():
        assert C._linear(layer, x).grad_fn is None


# outputs of 8, 4, 2 ranges and of one product; rows that do not divide
@pytest.mark.parametrize("rows,n,k", [(8192, 1536, 256), (8192, 2048, 2048), (8192, 6144, 1024), (8192, 6144, 2048), (8203, 512, 512)])
def test_a_hooked_layer_forms_its_weight_gradients_like_a_plain_one(rows, n, k):
    from lookahead_keys_attention_amd import castle as C

    torch.manual_seed(6)
    layer = torch.nn.Linear(k, n, bias=False).to(DEV).bfloat16()
    x = torch.randn(1, rows, k, device=DEV).bfloat16()
    gy = torch.randn(1, rows, n, device=DEV).bfloat16()
    y = C._linear(layer, x)
    assert "ManyRowLinear" in type(y.grad_fn).__name__
    y.backward(gy)
    assert torch.equal(layer.weight.grad, torch.ops.castle_hip.linear_bwd(gy, x, layer.weight.detach(), False, True)[1])
    ref = gy[0].float().t() @ x[0].float()
    assert (layer.weight.grad.float() - ref).norm() <= 4e-3 * ref.norm()   # one rounding to bf16
    handle = layer.register_forward_hook(lambda *_: None)   # on the projection itself: the module runs
    assert "ManyRowLinear" not in type(C._linear(layer, x).grad_fn).__name__
    handle.remove()
    # traced: a norm that is hooked keeps the layer from being taken apart into the library's operators
    norm = torch.nn.RMSNorm(k).to(DEV).bfloat16()
    norm.register_forward_hook(lambda *_: None)
    want = torch.autograd.grad(C._linear(layer, norm(x)), layer.weight, gy)[0]
    torch._dynamo.reset()
    traced = torch.compile(lambda t: C._linear(layer, norm(t)), backend="aot_eager", fullgraph=True)
    assert torch.equal(torch.autograd.grad(traced(x), layer.weight, gy)[0], want)
    # with a graph of the backward pass the gradient has derivatives
    leaf = x[:, :, :].clone().requires_grad_()
    dw, = torch.autograd.grad(C._linear(layer, leaf).sum(), layer.weight, create_graph=True)
    assert torch.autograd.grad(dw.sum(), leaf)[0].eq(n).all()


def test_dense_modules_over_many_rows_use_no_native_operator():
    from torch.utils._python_dispatch import TorchDispatchMode

    from lookahead_keys_attention_amd import CastleLM

    class NoNative(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            assert func.namespace != "castle_hip", func
            return func(*args, **(kwargs or {}))

    model = CastleLM(num_tokens=64, dim=32, depth=1, dim_head=16, heads=2, use_triton=False).to(DEV).bfloat16()
    with NoNative():
        model(torch.zeros(512, 17, dtype=torch.long, device=DEV), return_loss=True).backward()


@pytest.mark.parametrize("prenorm", [False, True])
def test_input_changed_in_place_before_the_backward_pass(prenorm):
    """A layer's input is read by its backward pass: one that was changed in place is an error, as for the modules
    one by one, where a gradient needs it, and no error where none does."""
    m = make(64, 2, 32, prenorm=prenorm)
    for wide in (False, True):   # rows of the input itself, and of a wider tensor
        h = torch.randn(2, 40, 80 if wide else 64, device=DEV)[..., :64]
        y = m(h)
        h += y.detach()
        if prenorm and wide:   # (the norm works on a copy of such rows)
            y.sum().backward()
            continue
        with pytest.raises(RuntimeError, match="modified by an inplace operation"):
            y.sum().backward()
    m.to_all_qkv.weight.requires_grad_(False)
    leaf = torch.randn(2, 40, 64, device=DEV, requires_grad=True)
    want, = torch.autograd.grad(m(leaf).sum(), leaf)
    h = leaf * 1
    y = m(h)
    h += 1
    if prenorm:
        with pytest.raises(RuntimeError, match="modified by an inplace operation"):
            y.sum().backward()
    else:   # no gradient reads the input of a frozen projection
        assert torch.equal(torch.autograd.grad(y.sum(), leaf)[0], want)


@pytest.mark.parametrize("dtype,tol", [(torch.bfloat16, 2e-2), (torch.float16, 4e-3)])
def test_step_and_parallel_pass_normalise_small_rows_alike(dtype, tol):
    """A norm without an eps of its own adds that of the 32-bit sums, whatever the type of the rows: with rows of 0.05 the
    type's epsilon would be three times their mean square.  (Tolerance: the types' roundings, as for the other steps.)"""
    from lookahead_keys_attention_amd import CastleLM

    m = make(128, 2, 64, dtype=dtype, prenorm=True).eval()
    x = torch.randn(2, 40, 128, generator=torch.Generator().manual_seed(8)).to(DEV).to(dtype)
    ids = torch.randint(0, 64, (2, 40), generator=torch.Generator().manual_seed(9)).to(DEV)
    lm = CastleLM(num_tokens=64, dim=128, depth=2, dim_head=64, heads=2).to(DEV).to(dtype).eval()
    with torch.no_grad():
        lm.token_emb.weight.mul_(0.02)
        for p in (lm.layers[0][0].combine_heads, lm.layers[0][1][3], lm.layers[1][0].combine_heads, lm.layers[1][1][3]):
            p.weight.mul_(0.02)   # the residual stream stays small
        for model, rows in ((m, x), (m, x * 0.05), (lm, ids)):
            want = model(rows)[:, -1]
            _, cache = model(rows[:, :39], return_next_cache=True)
            got = model(rows[:, 39:], cache=cache, return_next_cache=True)[0][:, 0]
            assert (got - want).double().norm() <= tol * want.double().norm()


@pytest.mark.parametrize("prenorm", [False, True])
def test_second_derivatives_of_a_layer_raise(prenorm):
    m = make(64, 2, 32, prenorm=prenorm)
    x = torch.randn(2, 40, 64, device=DEV, requires_grad=True)
    for leaf in (x, m.to_all_qkv.weight, m.combine_heads.weight):
        y = m(x)
        first, = torch.autograd.grad(y.square().sum(), leaf, create_graph=True)
        with pytest.raises(RuntimeError, match="differentiate twice"):
            (y.sum() + first.square().sum()).backward()
        assert torch.equal(first, torch.autograd.grad(m(x).square().sum(), leaf)[0])


@pytest.mark.parametrize("name", ["norm", "to_all_qkv", "combine_heads"])
def test_replaced_forward_and_traced_hooks_run(name):
    m = make(64, 2, 32, prenorm=True)
    x = torch.randn(2, 40, 64, device=DEV)
    layer, calls = getattr(m, name), []
    original = layer.forward

    def halved(t):
        calls.append(t.shape)
        return original(t) * 0.5

    with torch.no_grad():
        layer.forward = halved
        y, cache = m(x, return_next_cache=True)
        step, _ = m(x[:, :1], cache=cache)
        del layer.forward
        assert len(calls) == 2
        handle = layer.register_forward_hook(lambda module, args, out: out * 0.5)
        assert (m(x) - y).norm() <= 1e-5 * y.norm()
        compiled = torch.compile(m, backend="aot_eager")(x)
        assert (compiled - y).norm() <= 1e-5 * y.norm()
        handle.remove()
        layer.weight.mul_(0.5)   # the same in the weights
        y2, cache = m(x, return_next_cache=True)
        assert (y - y2).norm() <= 1e-5 * y2.norm() and (step - m(x[:, :1], cache=cache)[0]).norm() <= 1e-5 * step.norm()


def test_memory_of_a_dropped_cache_waits_for_a_step_on_another_stream():
    m = make(256, 4, 64, dtype=torch.bfloat16).eval()
    x = torch.randn(2, 70, 256, device=DEV).bfloat16()
    side = torch.cuda.Stream()
    with torch.no_grad():
        _, cache = m(x, return_next_cache=True)
        _, cache = m(x[:, :1], cache=cache)   # the step's scratch is allocated here
        want, _ = m(x[:, 1:2], cache=m(x[:, :1], cache=m(x, return_next_cache=True)[1])[1])
        store = cache._store
        kept = [*store.buffers, *store.rings, store.workspace]
        taken = {t.data_ptr() for t in kept}
        sizes = [t.numel() * t.element_size() for t in kept]
        projection = 2 * 6 * 4 * 64 * 2
        torch.cuda.synchronize()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            torch.cuda._sleep(20_000_000)   # (cycles of a clock of 100 MHz)
            got, cache = m(x[:, 1:2], cache=cache)
        del cache, store, kept
        fresh = [torch.empty(n, dtype=torch.uint8, device=DEV) for n in sizes]
        stats = torch.cuda.memory_stats()
        busy = not side.query()
        pending = stats["active_bytes.all.current"] - stats["allocated_bytes.all.current"]
    assert busy, "the step on the other stream was through before the check"
    assert not taken & {t.data_ptr() for t in fresh} and pending >= sum(sizes) + projection
    torch.cuda.synchronize()
    assert torch.equal(got, want)


def test_first_cached_step_recorded_into_a_graph():
    """A cache whose first step is recorded: steps outside the graph before its first replay, and replays between them, give what steps without a
    graph give (the recorded step must not prepare memory that those steps rely on)."""
    m = make(128, 2, 64, torch.bfloat16, prenorm=True).eval()
    g = torch.Generator(device=DEV).manual_seed(3)
    prompt, tokens = (torch.randn(2, n, 128, generator=g, device=DEV).bfloat16() for n in (20, 3))
    tokens = [tokens[:, i:i + 1].contiguous() for i in range(3)]
    with torch.no_grad():
        _, cache = m(prompt, return_next_cache=True)
        want = []
        for token in tokens:
            y, cache = m(token, cache=cache)
            want.append(y)
        _, cache = m(prompt, return_next_cache=True)
        store = cache._store
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            recorded, _ = m(tokens[0], cache=cache)
        store.length = 20   # recorded, not taken
        cache = store.as_cache()
        for i, token in enumerate(tokens):
            y, cache = m(token, cache=cache)
            assert torch.equal(y, want[i]) if i == 0 else True
            bf16_close(y, want[i], f"step {i}")
            if i < 2:   # (the step at 20 again; the lookahead keys are written at 23 only)
                recorded.fill_(7)
                graph.replay()
                torch.cuda.synchronize()
                bf16_close(recorded, want[0], f"replay {i}")


def test_control_words_only_for_caches_whose_steps_go_in_one_launch():
    """What a first step keeps for later ones: its projection, and control words where it is one launch."""
    from lookahead_keys_attention_amd import _native as N

    for B, heads, n in ((1, 8, 100), (16, 16, 40), (8, 8, 1000)):
        m = make(512, heads, 64, torch.bfloat16).eval()
        lib, inner = N.lib(), heads * 64
        with torch.no_grad():
            x = torch.randn(B, n, 512, device=DEV).bfloat16()
            _, cache = m(x, return_next_cache=True)
            cache._store.workspace
            token = x[:, :1].contiguous()
            y = m(token)   # whatever a first step of all allocates
            y = None
            before = torch.cuda.memory_allocated()
            y, cache = m(token, cache=cache)
            kept = torch.cuda.memory_allocated() - before
        up = lambda n: (n + 511) // 512 * 512
        once = lib.castle_decode_layer_once_ok(B, heads, 64, 1, n, 512)
        assert once == (B == 1)
        control = lib.castle_decode_layer_control_bytes(B, heads, 64, 1) if once else 0
        assert kept == up(B * 6 * inner * 2) + up(y.numel() * 2) + up(control)


def test_forward_mode_derivatives_of_a_layer_raise():
    from torch.autograd import forward_ad

    m = make(64, 2, 32).requires_grad_(False)
    x = torch.randn(2, 40, 64, device=DEV)
    for rows in (x, x[:, :1]):   # the parallel pass, a cached step
        with forward_ad.dual_level(), pytest.raises(NotImplementedError, match="forward-mode"):
            m(forward_ad.make_dual(rows, torch.ones_like(rows)))


def test_multi_token_with_cache_is_rejected():
    m = make(32, 2, 16)
    x = torch.randn(1, 4, 32).to(DEV)
    _, cache = m(x, return_next_cache=True)
    with pytest.raises(AssertionError):
        m(x, cache=cache)


def test_auto_selected_kernels_leave_uncovered_shapes_to_the_dense_path():
    """use_triton=None (the reference's default, lookahead_keys_attention.py:58) picks the kernels where
    they apply and the PyTorch formulation elsewhere: a head dimension or tensor type the kernels do
    not cover still runs (forward, backward, cached steps == parallel), while an explicit
    use_triton=True on the same module raises."""
    from lookahead_keys_attention_amd import Castle

    torch.manual_seed(3)
    for d, dtype in ((48, torch.float32), (128, torch.float32), (32, torch.float64)):
        m = Castle(64, heads=2, dim_head=d, use_triton=None).to(DEV).to(dtype)
        assert m.use_triton   # the kernels are built and a GPU is there; this shape is simply not theirs
        x = torch.randn(2, 9, 64, device=DEV, dtype=dtype, requires_grad=True)
        y, cache = m(x, return_next_cache=True)
        y.sum().backward()
        assert torch.isfinite(x.grad).all()
        with torch.no_grad():
            full = m(torch.cat([x.detach(), x.detach()[:, :1]], dim=1))
            step, _ = m(x.detach()[:, :1], cache=cache)
        assert torch.allclose(step[:, 0], full[:, -1], atol=1e-4)
        explicit = Castle(64, heads=2, dim_head=d, use_triton=True).to(DEV).to(dtype)
        with pytest.raises((ValueError, TypeError, RuntimeError)):
            explicit(x.detach())


def test_config1_readme_fp32_parallel_vs_sequential():
    # benchmark configuration 1: Castle(512, 8, 64), x (2,128,512) fp32, parallel vs 128 cached steps, atol 1e-3
    m = make(512, 8, 64, seed=0).eval()
    x = torch.randn(2, 128, 512, generator=torch.Generator().manual_seed(0))
    with torch.no_grad():
        full = m(x.to(DEV))
        cache, ys = None, []
        for t in range(128):
            y, cache = m(x[:, t:t + 1].to(DEV), cache=cache)
            ys.append(y)
    seq = torch.cat(ys, 1)
    assert (seq - full).abs().max() <= 1e-3
    ref = O.module_forward(x, cpu_params(m), 8)
    assert (full.cpu() - ref).abs().max() <= 1e-3 and (seq.cpu() - ref).abs().max() <= 1e-3


def _head_oracle_check(proj, dmerged, merged, dproj, heads, d, b, h, nb=None, dtype=torch.float32):
    """Oracle for one (b, h) slice of a packed bf16 run: out and the six gradients.  nb=None takes the
    dense formulation (parallel_core, closed_form_grads), else the streamed state forms with row blocks
    of nb (blockwise_head: pinned against the dense ones in tests/test_oracle_core.py), which reach
    full-length heads."""
    B, L, _ = proj.shape
    six = proj.view(B, L, 6, heads, d)
    qu, ku, vu, qc, kc, vc = [six[b, :, i, h].to(dtype).cpu() for i in range(6)]
    do = dmerged.view(B, L, heads, d)[b, :, h].to(dtype).cpu()
    s = d ** -0.5
    if nb is None:
        out = O.parallel_core(qc, kc, vc, qu, ku, vu, s)
        grads = O.closed_form_grads(qc, kc, vc, qu, ku, vu, s, do)
    else:
        out, _, grads = O.blockwise_head(qc, kc, vc, qu, ku, vu, s, nb, do)
    bf16_close(merged.view(B, L, heads, d)[b, :, h], out, f"out[{b},{h}]")
    g6 = dproj.view(B, L, 6, heads, d)
    for name, idx, r in zip(("dqc", "dkc", "dvc", "dqu", "dku", "dvu"), (3, 4, 5, 0, 1, 2), grads):
        bf16_close(g6[b, :, idx, h], r, f"{name}[{b},{h}]")


def test_config2_bf16_full_size_sampled_heads():
    # benchmark configuration 2: dim 512, H8, d64, B4, L4096, bf16, forward + backward
    from lookahead_keys_attention_amd import ops

    m = make(512, 8, 64, dtype=torch.bfloat16, seed=0)
    g = torch.Generator().manual_seed(0)
    x = torch.randn(4, 4096, 512, generator=g).bfloat16().to(DEV)
    gy = torch.randn(4, 4096, 512, generator=g).bfloat16().to(DEV)
    proj = m.to_all_qkv(x).detach().requires_grad_()
    merged = ops.castle_attention_packed(proj, 8, m.scale)
    dmerged = (gy @ m.combine_heads.weight.detach())
    merged.backward(dmerged)
    assert torch.isfinite(merged).all() and torch.isfinite(proj.grad).all()
    # eight (b, h) slices, one per value of (b * 8 + h) % 8: the kernels keep head bh on XCD bh % 8,
    # so every XCD's share is checked; two of them also against the dense formulation
    for b, h in ((0, 0), (1, 1), (2, 2), (3, 3), (0, 4), (3, 5), (2, 6), (1, 7)):
        _head_oracle_check(proj.detach(), dmerged, merged.detach(), proj.grad, 8, 64, b, h, nb=256, dtype=torch.float64)
    for b, h in ((0, 0), (3, 5)):
        _head_oracle_check(proj.detach(), dmerged, merged.detach(), proj.grad, 8, 64, b, h)
    # causality at full size: the first 1024 positions do not depend on the rest
    short = ops.castle_attention_packed(proj.detach()[:, :1024].contiguous(), 8, m.scale)
    bf16_close(merged.detach()[:, :1024], short, "prefix invariance")


def test_config3_bf16_long_context_forward_backward():
    # benchmark configuration 3: dim 2048, H16, d128, B1, L16384, bf16, forward + backward at full size.
    # The dense oracle at L=16384 is out of reach on CPU; the streamed state form of the oracle is not:
    # (o) two heads of the full-length run, forward and all six gradients, against oracle.blockwise_head
    # in fp32 (lookahead scores have a standard deviation of about 20 at this length).  Beside it,
    # size-independent properties: (i) prefix invariance of the forward output; (iii) the backward
    # pass is linear in dO, and positions whose dO is zero (and that no later position with a
    # non-zero dO exists for) get exactly zero query/key/value gradients; and (ii) the same operator
    # on the first 2048 positions is compared with the dense oracle (one head).
    from lookahead_keys_attention_amd import ops

    m = make(2048, 16, 128, dtype=torch.bfloat16, seed=0)
    g = torch.Generator().manual_seed(0)
    x = torch.randn(1, 16384, 2048, generator=g).bfloat16().to(DEV)
    gy = torch.randn(1, 16384, 2048, generator=g).bfloat16().to(DEV)
    with torch.no_grad():
        proj = m.to_all_qkv(x)
        dmerged = gy @ m.combine_heads.weight.detach()
    leaf = proj.clone().requires_grad_()
    merged = ops.castle_attention_packed(leaf, 16, m.scale)
    merged.backward(dmerged)
    g1 = leaf.grad.clone()
    assert torch.isfinite(merged).all() and torch.isfinite(g1).all()
    # (o) full-length heads against the streamed oracle
    for h in (7, 12):
        _head_oracle_check(proj, dmerged, merged.detach(), g1, 16, 128, 0, h, nb=256)
    # (i) prefix invariance of the forward
    with torch.no_grad():
        short = ops.castle_attention_packed(proj[:, :2048].contiguous(), 16, m.scale)
    bf16_close(merged.detach()[:, :2048], short, "prefix invariance")
    # (iii) linearity of the backward in dO: grad(2 dO) == 2 grad(dO), bit for bit up to bf16 rounding
    leaf2 = proj.clone().requires_grad_()
    ops.castle_attention_packed(leaf2, 16, m.scale).backward(dmerged * 2)
    bf16_close(leaf2.grad, g1.float() * 2, "linearity in dO")
    # a zero upstream gradient on the last 4096 positions leaves their operands' query-side gradients zero
    dm0 = dmerged.clone()
    dm0[:, 12288:] = 0
    leaf3 = proj.clone().requires_grad_()
    ops.castle_attention_packed(leaf3, 16, m.scale).backward(dm0)
    g3 = leaf3.grad.view(1, 16384, 6, 16, 128)
    assert torch.all(g3[:, 12288:, 3] == 0)          # dqc of positions whose dO is zero
    assert torch.all(g3[:, 12288:, 4:6] == 0)        # keys/values only they (and later) could see: dkc, dvc
    # (ii) L = 2048 slice against the oracle, forward and backward, one head
    leaf4 = proj[:, :2048].clone().requires_grad_()
    out4 = ops.castle_attention_packed(leaf4, 16, m.scale)
    out4.backward(dmerged[:, :2048].contiguous())
    _head_oracle_check(leaf4.detach(), dmerged[:, :2048].contiguous(), out4.detach(), leaf4.grad, 16, 128, 0, 7)


def test_config4_bf16_decode_after_prefill():
    """benchmark configuration 4 at full size: B32, prefill 2048 through the parallel path, then all
    512 cached steps with fresh x_t ~ N(0,1).  The native decode's per-head output (before the
    output projection) of sampled (b, h) is compared at steps 1, 256 and 512 with the oracle's
    decode_core iterated in fp32 on that head from the oracle's own prefill (nothing of the native
    step's rounding cadence is imitated), and so are the head's lookahead keys in the cache after the
    last step.  The reference's step forms `U = U_prev + gate * vu` in the module dtype
    (lookahead_keys_attention.py:183): in bf16 that is 512 roundings of every row to 8 significant
    bits, and its last step then differs from its own parallel pass by about 5e-2 normwise.  The native
    cache writes the keys back on every 4th step and holds them with 11 significant bits, so parallel
    and sequential agree inside the 2e-2 rule."""
    m = make(512, 8, 64, dtype=torch.bfloat16, seed=0).eval()
    g = torch.Generator().manual_seed(0)
    steps, t0 = 512, 2048
    x = torch.randn(32, t0 + steps, 512, generator=g).bfloat16().to(DEV)
    heads = [(17, 3), (0, 0), (31, 7)]
    watch = {1, 256, 512}
    native = {}
    with torch.no_grad():
        proj_all = m.to_all_qkv(x).view(32, t0 + steps, 6, 8, 64)
        _, cache = m(x[:, :t0], return_next_cache=True)
        for n in range(1, steps + 1):
            t = t0 + n - 1
            merged, cache = m._step_native(m.to_all_qkv(x[:, t:t + 1]), cache)
            if n in watch:
                native[n] = merged.view(32, 8, 64).float().cpu()
        # the module's own step (projection included) agrees with the parallel pass on the last row
        full_last = m(x)[:, -1]
    assert cache.U.shape == (32, 8, t0 + steps, 64) and cache.U.dtype == torch.bfloat16
    last = m.combine_heads(merged)[:, 0].double().cpu()
    drift = ((last - full_last.double().cpu()).norm() / full_last.double().norm()).item()
    worst = ((last - full_last.double().cpu()).abs().max() / full_last.double().abs().max()).item()
    assert drift <= 2e-2 and worst <= 2e-2, f"last cached step vs parallel: {drift:.3e} normwise, {worst:.3e} of max"
    gotU_all = cache.U
    for b, h in heads:
        qu, ku, vu, qc, kc, vc = [proj_all[b, :, i, h].float().cpu() for i in range(6)]
        _, U0 = O.parallel_core(*[t[:t0] for t in (qc, kc, vc, qu, ku, vu)], m.scale, want_U=True)
        state = (U0, qu[:t0], kc[:t0], vc[:t0])
        for n in range(1, steps + 1):
            t = t0 + n - 1
            out, state = O.decode_core(state, *[z[t:t + 1] for z in (qc, kc, vc, qu, ku, vu)], m.scale)
            if n in watch:
                bf16_close(native[n][b, h], out[0], f"decode step {n} of head ({b},{h}) vs oracle")
        bf16_close(gotU_all[b, h], state.U, f"lookahead keys of head ({b},{h}) after {steps} steps")
        assert torch.equal(cache.kc_cache[b, h].float().cpu(), kc) and torch.equal(cache.qu_cache[b, h].float().cpu(), qu)
