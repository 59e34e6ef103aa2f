"""Row kernels (norm with a residual sum, cross entropy, embedding gradient) against fp32 / fp64 PyTorch on the CPU."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
TOL = {torch.float32: 2e-5, torch.bfloat16: 1e-2, torch.float16: 2e-3}


def host():
    from lookahead_keys_attention_amd import _native

    return _native.host()


def close(got, ref, dtype, what):
    got, ref = got.detach().cpu().double(), ref.detach().double()
    assert torch.isfinite(got).all() and (got - ref).norm() <= TOL[dtype] * ref.norm() + 1e-30, (what, (got - ref).norm() / ref.norm())


# lanes per row 16 / 32 / 64, 1 ... 8 pieces per lane, their edges, a length for the library's norm (5000)
@pytest.mark.parametrize("dim", [8, 120, 128, 136, 256, 512, 520, 1024, 2048, 4096, 5000])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32, torch.float16])
def test_norm_with_sum(dim, dtype):
    g = torch.Generator().manual_seed(dim)
    for B, L in ((1, 2), (3, 43), (2, 1500 if dim <= 512 else 60)):
        x, delta, gy = (torch.randn(B, L, n, generator=g).to(dtype) for n in (dim, dim, 16))
        nw, w = (1 + torch.randn(dim, generator=g) * 0.2).to(dtype), (torch.randn(16, dim, generator=g) * dim ** -0.5).to(dtype)
        leaves = [t.to(DEV).requires_grad_() for t in (x, delta, nw, w)]
        y = host().head(leaves[0], leaves[1], leaves[2], None, leaves[3])
        y.backward(gy.to(DEV))
        ref = [t.double().requires_grad_() for t in (x, delta, nw, w)]
        s = ref[0] + ref[1]
        yr = F.rms_norm(s + ((x + delta).double() - s).detach(), (dim,), ref[2], torch.finfo(torch.float32).eps) @ ref[3].t()
        yr.backward(gy.double())
        close(y, yr, dtype, "y")
        for name, a, b in zip(("x", "delta", "norm", "w"), leaves, ref):
            close(a.grad, b.grad, dtype, name)
        with torch.no_grad():
            assert torch.equal(host().head(*leaves[:3], None, leaves[3]), y)


@pytest.mark.parametrize("classes", [8, 256, 264, 1000, 32000])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_cross_entropy(classes, dtype):
    g = torch.Generator().manual_seed(classes)
    for B, n in ((1, 1), (3, 37), (5, 1100 if classes <= 256 else 20)):
        logits = (torch.randn(B, n, classes, generator=g) * 3).to(dtype)
        target = torch.randint(0, classes, (B, n + 1), generator=g)
        if n > 1:
            target[0, 1] = -100
        leaf = logits.to(DEV).requires_grad_()
        loss = host().cross_entropy(leaf, target.to(DEV)[:, 1:])
        (loss * 2).backward()
        ref = logits.double().requires_grad_()
        lr = F.cross_entropy(ref.transpose(1, 2), target[:, 1:]) if n > 1 or target[0, 1] != -100 else None
        (lr * 2).backward()
        close(loss, lr, dtype, "loss")
        close(leaf.grad, ref.grad, dtype, "dlogits")
    bad = target.clone()
    bad[0, 2] = classes
    assert host().cross_entropy(leaf.detach(), bad.to(DEV)[:, 1:]).isnan()


@pytest.mark.parametrize("classes", [8, 256, 1000])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_cross_entropy_of_nan_and_infinite_logits(classes, dtype):
    """One NaN, an aligned 16-byte piece of them, a whole row; infinities of either sign: like the library on the CPU."""
    piece, inf, nan = 16 // dtype.itemsize, float("inf"), float("nan")
    g = torch.Generator().manual_seed(classes)
    base, target = torch.randn(1, 5, classes, generator=g).to(dtype), torch.randint(0, classes, (1, 5), generator=g)
    last = classes - piece
    for where, value in ((slice(0, 1), nan), (slice(0, piece), nan), (slice(last, classes), nan), (slice(0, classes), nan), (slice(0, piece), -inf),
                         (slice(0, classes), -inf), (slice(0, 1), inf), (slice(0, classes), inf)):
        logits = base.clone()
        logits[0, 2, where] = value
        if value == -inf and classes > piece:
            target[0, 2] = last   # (a class that is not among them)
        leaf, ref = logits.to(DEV).requires_grad_(), logits.double().requires_grad_()
        loss, want = host().cross_entropy(leaf, target.to(DEV)), F.cross_entropy(ref.transpose(1, 2), target)
        assert loss.isnan() == want.isnan().to(DEV) and (want.isnan() or (loss.cpu().double() - want).abs() <= TOL[dtype] * want.abs())
        loss.backward()
        want.backward()
        assert torch.equal(leaf.grad.isnan().cpu(), ref.grad.isnan())
        finite = ~ref.grad.isnan()
        close(leaf.grad.cpu()[finite], ref.grad[finite], dtype, "dlogits")
        # a row that does not count brings nothing in
        target_without = target.clone()
        target_without[0, 2] = -100
        leaf.grad = None
        loss = host().cross_entropy(leaf, target_without.to(DEV))
        loss.backward()
        assert loss.isfinite() and leaf.grad.isfinite().all() and not leaf.grad[0, 2].any()


def test_cross_entropy_of_a_class_out_of_range():
    logits = torch.randn(2, 3, 264, device=DEV).requires_grad_()
    for bad in (264, -1, 1 << 40, -(1 << 40)):
        target = torch.tensor([[1, 2, 3], [4, bad, -100]], device=DEV)
        loss = host().cross_entropy(logits, target)
        grad, = torch.autograd.grad(loss, logits)
        assert loss.isnan() and grad[1, 1].isnan().all() and grad[0].isfinite().all() and not grad[1, 2].any()


@pytest.mark.parametrize("vocabulary,dim", [(5, 8), (256, 512), (300, 1032)])
def test_embedding_gradient(vocabulary, dim):
    g = torch.Generator().manual_seed(vocabulary)
    for B, n in ((1, 1), (2, 1025), (3, 2048)):
        w, ids = torch.randn(vocabulary, dim, generator=g).bfloat16(), torch.randint(0, vocabulary, (B, n + 1), generator=g)
        ids[0] = 1   # one row gets most of them
        dy = torch.randn(B, n, dim, generator=g).bfloat16()
        leaf = w.to(DEV).requires_grad_()
        y = host().embedding(leaf, ids.to(DEV)[:, :-1])
        y.backward(dy.to(DEV))
        ref = w.double().requires_grad_()
        F.embedding(ids[:, :-1], ref).backward(dy.double())
        assert torch.equal(y.cpu(), F.embedding(ids[:, :-1], w))
        close(leaf.grad, ref.grad, torch.bfloat16, "dw")


def test_language_model_blocks_equal_the_modules():
    """The one-call-per-block path against the same model run module by module (a hook switches it off)."""
    from lookahead_keys_attention_amd import CastleLM

    torch.manual_seed(0)
    for tie in (False, True):
        model = CastleLM(num_tokens=64, dim=128, depth=2, heads=2, dim_head=64, tie_embedding=tie).to(DEV)
        ids = torch.randint(0, 64, (3, 90), device=DEV)
        results = []
        for hooked in (False, True):
            handle = model.layers[1][1].register_forward_hook(lambda *_: None) if hooked else None
            assert model._plain(ids) is not hooked
            model.zero_grad()
            loss = model(ids, return_loss=True)
            loss.backward()
            with torch.no_grad():
                logits, caches = model(ids, return_next_cache=True)
            results.append([loss, logits, caches[1].vc_cache] + [p.grad for p in model.parameters() if p.grad is not None])
            if handle is not None:
                handle.remove()
        assert len(results[0]) == len(results[1])
        for a, b in zip(*results):
            assert (a - b).norm() <= 1e-4 * b.norm()


def test_gradients_beside_caches_equal_those_without():
    """The nodes' outputs are y, the running sum and the rows of a cache, in any combination."""
    from lookahead_keys_attention_amd import CastleLM

    torch.manual_seed(0)
    model = CastleLM(num_tokens=64, dim=64, depth=2, heads=2, dim_head=32).to(DEV)
    ids = torch.randint(0, 64, (2, 40), device=DEV)
    params = [p for p in model.parameters() if p.requires_grad]
    results = []
    for cached in (False, True):
        out = model(ids, return_next_cache=cached)
        results.append(torch.autograd.grad((out[0] if cached else out).square().sum(), params))
    assert all(torch.equal(a, b) for a, b in zip(*results))


def test_replaced_forward_in_a_language_model_runs():
    from lookahead_keys_attention_amd import CastleLM

    torch.manual_seed(0)
    model = CastleLM(num_tokens=64, dim=64, depth=2, heads=2, dim_head=32).to(DEV)
    ids = torch.randint(0, 64, (2, 40), device=DEV)
    attention, feed_forward = model.layers[1]
    for module in (model.token_emb, attention, attention.norm, feed_forward, feed_forward[0], feed_forward[1], feed_forward[2], feed_forward[3],
                   model.final_norm, model.to_logits):
        assert model._plain(ids)
        calls, original = [], module.forward

        def counted(*args, **kwargs):
            calls.append(1)
            return original(*args, **kwargs)

        module.forward = counted
        assert not model._plain(ids)
        model(ids, return_loss=True)
        assert len(calls) == 1
        model.sample(ids[:, :6], 6 + 12)   # a prompt, eleven steps
        assert len(calls) == 1 + 12
        kept = model.__dict__.get("_kept_decoder")
        if module is attention:
            with pytest.raises(RuntimeError, match="would not run"):
                model.sample(ids[:, :6], 6 + 12, graph=True)
        else:   # insisted on: what the module does is captured, for this call
            model.sample(ids[:, :6], 6 + 12, graph=True)
            assert len(calls) > 1 + 12 and model.__dict__.get("_kept_decoder") is kept
        del module.forward
        model.sample(ids[:, :6], 6 + 12)
        assert model._kept_decoder is not None and (kept is None or model._kept_decoder is kept)


def test_subclasses_of_the_attention_layer_in_a_sampled_model():
    """One that leaves `forward` alone is captured like the layer itself; one that has its own is stepped."""
    from lookahead_keys_attention_amd import Castle, CastleLM

    class Named(Castle):
        pass

    class Counted(Castle):
        calls = 0

        def forward(self, *args, **kwargs):
            Counted.calls += 1
            return super().forward(*args, **kwargs)

    torch.manual_seed(0)
    model = CastleLM(num_tokens=64, dim=64, depth=2, heads=2, dim_head=32).to(DEV)
    ids = torch.randint(0, 64, (2, 6), device=DEV)
    want = model.sample(ids, 6 + 12, temperature=0)
    for kind, kept in ((Named, True), (Counted, False)):
        model.release_decoder()
        model.layers[1][0].__class__ = kind
        assert torch.equal(model.sample(ids, 6 + 12, temperature=0), want)
        assert ("_kept_decoder" in model.__dict__) == kept
    assert Counted.calls == 12


def test_second_derivatives_of_the_language_model_blocks_raise():
    """Every parameter's gradient: embedding, attention, feed-forward, head and loss are nodes of their own."""
    from lookahead_keys_attention_amd import CastleLM

    torch.manual_seed(0)
    model = CastleLM(num_tokens=64, dim=64, depth=2, heads=2, dim_head=32).to(DEV)
    ids = torch.randint(0, 64, (2, 40), device=DEV)
    assert model._plain(ids)
    for name, p in model.named_parameters():
        if p.requires_grad:
            loss = model(ids, return_loss=True)
            grad, = torch.autograd.grad(loss, p, create_graph=True)
            with pytest.raises(RuntimeError, match="differentiate twice"):
                (loss + grad.square().sum()).backward()


# tiles of 64 and 128 with remainders in every direction, contractions of less than a step, ranges of the contraction
@pytest.mark.parametrize("rows,n,k", [(1, 8, 8), (63, 72, 40), (65, 128, 200), (96, 768, 128), (257, 1536, 264), (1003, 256, 2048), (3000, 520, 512),
                                      (4500, 2048, 512)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32, torch.float16])
def test_products(rows, n, k, dtype):
    g = torch.Generator(device=DEV).manual_seed(rows)
    x, w, dy = (torch.randn(*s, generator=g, device=DEV).to(dtype) for s in ((rows, k), (n, k), (rows, n)))
    tol = {torch.float32: 1e-5, torch.bfloat16: 4e-3, torch.float16: 6e-4}[dtype]

    def check(got, ref, what):
        assert torch.isfinite(got).all() and (got.double() - ref).norm() <= tol * ref.norm(), (what, (got.double() - ref).norm() / ref.norm())

    wide = torch.full((rows, k + 16), 3.0, device=DEV, dtype=dtype)
    wide[:, :k] = x   # rows of a wider tensor
    ref = x.double() @ w.double().t()
    check(host().product(wide[:, :k], False, w, False, 0, None), ref, "forward")
    check(host().product(dy, False, w, True, 0, None), dy.double() @ w.double(), "input gradient")
    if n % 8 == 0:
        check(host().product(dy, True, x, True, 0, None), dy.double().t() @ x.double(), "weight gradient")
    act = torch.empty(rows, n, device=DEV, dtype=dtype)
    up = host().product(x, False, w, False, 1, act)
    assert torch.equal(up, host().product(x, False, w, False, 2, torch.full_like(act, 30.0)))   # the slope is 1 there
    check(act, F.gelu(up.double()), "gelu")
    u = torch.randn(rows, k, generator=g, device=DEV).to(dtype)
    plain = dy.double() @ w.double()
    slope = torch.autograd.functional.vjp(F.gelu, u.double(), torch.ones_like(plain))[1]
    check(host().product(dy, False, w, True, 2, u), plain * slope, "slope")


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rows,n,k", [(65, 72, 264), (130, 264, 328), (192, 64, 1000), (320, 512, 136), (456, 584, 520), (511, 456, 584)])
def test_products_of_two_groups(rows, n, k, dtype):
    """One tile a CU and a contraction of four steps and more (16-bit operands: eight): even and odd numbers of steps, a last one that is
    partly filled, one that only the first group has."""
    if rows > 400 and dtype == torch.bfloat16:   # in each layout; the others are so in some layouts, fp32 also in ranges of the contraction
        assert all(gemm_plan(*sizes, dtype, 0, groups=True) == 2 for sizes in ((rows, n, k), (rows, k, n), (n, k, rows)))
    test_products(rows, n, k, dtype)
    if dtype == torch.bfloat16 and (256 <= k < 512 or rows > 400):   # (split elsewhere, and no maxima are taken)
        test_product_leaves_partial_maxima(rows, n, k, 8, n - 16)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows,n,k", [(2112, 3136, 512), (2112, 512, 3136), (8136, 2040, 512), (8136, 512, 2040), (8136, 2040, 320), (4160, 3136, 448),
                                      (2112, 6144, 1024)])
def test_products_of_wide_tiles(rows, n, k, dtype):
    """Tiles of 256 x 128 and 256 x 256 in each layout: last ones of 64 rows and columns and of odd eights, even and odd numbers of steps,
    one tile a CU, ranges of the contraction."""
    test_products(rows, n, k, dtype)
    if dtype == torch.bfloat16 and n > k:
        test_product_leaves_partial_maxima(rows, n, k, 520, 256)


def gemm_plan(M, N, K, dtype, epilogue, groups=False):
    """(rows, columns) of a tile, and how many of them a launch has; or how many groups of waves share one."""
    import ctypes

    from lookahead_keys_attention_amd import _native

    out = [ctypes.c_int() for _ in range(4)]
    _native.check(_native.lib().castle_gemm_plan(M, N, K, _native.DTYPE_CODES[dtype], epilogue, *map(ctypes.byref, out)), "castle_gemm_plan")
    rows, columns, ranges, waves = (v.value for v in out)
    if groups:
        return waves
    return (rows, columns), -(-M // rows) * -(-N // columns) * ranges


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,N,K,plain,fused", [(16456, 1032, 512, (256, 128), None), (8456, 1992, 256, (256, 128), None), (16456, 1032, 64, (256, 128), None),
                                               (8456, 3064, 256, (256, 256), None), (8456, 3064, 128, (256, 256), None), (8456, 3064, 64, (256, 256), None),
                                               (8456, 3064, 512, (256, 256), (256, 256)), (16456, 2040, 512, (256, 256), (256, 128)),
                                               (16456, 4088, 64, (256, 128), (256, 128))])
def test_products_of_several_wide_tiles_a_workgroup(M, N, K, plain, fused, dtype):
    """More tiles of 256 rows than CUs, so that a workgroup goes on to the next while the last is being stored, between whole tiles and ones with remainders, of one
    step of the contraction, two and more, in each layout and with gelu, its slope and the maxima on the store.  Element by element: K products and sums of 2^-24 each, at most, and the roundings
    to the type (halves of fp16's smallest step, 2^-25, where the result is below its normal numbers); gelu of the rounded product to 2^-20 before its own."""
    g = torch.Generator(device=DEV).manual_seed(M + N)
    a, b, u = (torch.randn(*s, generator=g, device=DEV).to(dtype) for s in ((M, K), (N, K), (M, N)))
    ref, size, bits = a.double() @ b.double().t(), a.double().abs() @ b.double().abs().t(), {torch.bfloat16: 8, torch.float16: 11}[dtype]
    tiny = 2.0 ** -25 if dtype == torch.float16 else 0.0
    error = (K + 4) * 2.0 ** -24 * size + 2.0 ** -bits * ref.abs() + tiny
    layouts = [(a, False, b, False), (a, False, b.t().contiguous(), True), (a.t().contiguous(), True, b.t().contiguous(), True)]
    tile, tiles = gemm_plan(M, N, K, dtype, 0)
    assert tile == plain and tiles > 256
    for operands in layouts:
        assert torch.all((host().product(*operands, 0, None).double() - ref).abs() <= 1.01 * error)
    if dtype == torch.bfloat16:
        test_product_leaves_partial_maxima(M, N, K, 520, 256)
    if fused is None:
        return
    tile, tiles = gemm_plan(M, N, K, dtype, 1)
    assert tile == fused and tiles > 256
    v = u.double()
    slope = torch.special.ndtr(v) + v * torch.exp(-v * v / 2) / (2 * torch.pi) ** 0.5
    for operands in layouts:
        act = torch.empty_like(u)
        up = host().product(*operands, 1, act)
        assert torch.all((up.double() - ref).abs() <= 1.01 * error)
        gelu = F.gelu(up.double())
        assert torch.all((act.double() - gelu).abs() <= 1.01 * 2.0 ** -bits * gelu.abs() + 2.0 ** -20 * up.double().abs() + tiny)
        got = host().product(*operands, 2, u).double()
        over = (got - ref * slope).abs() - (1.01 * (slope.abs() * error + 2.0 ** -bits * (ref * slope).abs()) + 2.0 ** -18 * ref.abs() + tiny)
        at = over.argmax().item()
        assert over.max().item() <= 0, (over.max().item(), got.flatten()[at].item(), (ref * slope).flatten()[at].item(), ref.flatten()[at].item(), u.flatten()[at].item())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32, torch.float16])
@pytest.mark.parametrize("rows,n,k", [(1, 8, 8), (63, 72, 40), (96, 768, 128), (65, 264, 264), (130, 1536, 512), (200, 136, 456), (1000, 640, 1000), (70, 128, 248)])
def test_product_of_normalised_rows(rows, n, k, dtype):
    """Norm and product in one launch, with and without what a backward pass reads: remainders in every direction, one group of waves and two."""
    import ctypes

    from lookahead_keys_attention_amd import _native as N

    class Norm(ctypes.Structure):
        _fields_ = [("weight", ctypes.c_void_p), ("eps", ctypes.c_float), ("h", ctypes.c_void_p), ("rstd", ctypes.c_void_p)]

    lib, code = N.lib(), N.DTYPE_CODES[dtype]
    vp, i, i64 = ctypes.c_void_p, ctypes.c_int, ctypes.c_int64
    lib.castle_gemm_of_norm.argtypes = [vp, i64, ctypes.POINTER(Norm), vp, i64, vp, i64, i, i, i, i, vp, vp]
    if not lib.castle_gemm_norm_ok(rows, n, k, code):
        assert dtype is torch.float32   # a row too long, or a contraction that is better split
        return
    g = torch.Generator(device=DEV).manual_seed(rows)
    x, w, weight = (torch.randn(*s, generator=g, device=DEV).to(dtype) for s in ((rows, k + 8), (n, k), (k,)))
    x = (x * torch.logspace(-3, 2, rows, device=DEV)[:, None]).to(dtype)
    bits = {torch.float32: 24, torch.bfloat16: 8, torch.float16: 11}[dtype]
    factor = (x[:, :k].double().square().mean(dim=-1) + 1e-6).rsqrt()
    rows_ref = x[:, :k].double() * factor[:, None] * weight.double()
    out = []
    for keep in (True, False):
        c, h, rstd = torch.full((rows, n + 8), 7.0, device=DEV, dtype=dtype), torch.full((rows, k), 7.0, device=DEV, dtype=dtype), torch.full((rows,), 7.0, device=DEV)
        norm = Norm(weight.data_ptr(), 1e-6, h.data_ptr() if keep else None, rstd.data_ptr() if keep else None)
        N.check(lib.castle_gemm_of_norm(x.data_ptr(), k + 8, ctypes.byref(norm), w.data_ptr(), k, c.data_ptr(), n + 8, rows, n, k, code, None,
                                        N.stream_ptr(x.device)), "castle_gemm_of_norm")
        torch.cuda.synchronize()
        out.append(c)
        assert torch.all(c[:, n:] == 7)
        if keep:
            # (the factor: k squares and k sums of 2^-24 each, at most; halved by the root)
            assert torch.all((rstd.double() - factor).abs() <= (k + 4) * 2.0 ** -24 * factor)
            small = 2.0 ** -24 if dtype is torch.float16 else 0.0   # half of the smallest step
            assert torch.all((h.double() - rows_ref).abs() <= (2.0 ** -bits + (k + 8) * 2.0 ** -24) * rows_ref.abs() + small)
            ref = h.double() @ w.double().t()
            alone = torch.ops.castle_hip.rms_norm(x[:, :k].contiguous(), weight, 1e-6)   # the same bits as the norm by itself
            assert torch.equal(h, alone[0]) and torch.equal(rstd, alone[1])
    assert torch.equal(out[0], out[1])
    bound = (k + 4) * 2.0 ** -24 * (rows_ref.abs() @ w.double().abs().t()) + 2.0 ** -bits * ref.abs() + (2.0 ** -24 if dtype is torch.float16 else 0.0)
    assert torch.all((out[0][:, :n].double() - ref).abs() <= 1.01 * bound)


@pytest.mark.parametrize("k", [1, 63, 129, 257, 321])
def test_products_near_the_reach_of_32_bit_offsets(k):
    """A contraction over rows as far apart as the products take: two groups of waves step up to 382 rows behind its end."""
    import ctypes

    from lookahead_keys_attention_amd import _native as N

    ld, ok = ((1 << 31) // (k + 192) - 1) // 8 * 8, N.lib().castle_gemm_operand_ok
    ok.argtypes = [ctypes.c_int64] * 2
    assert ok(k, ld) and not ok(k, ld + 16)
    g = torch.Generator(device=DEV).manual_seed(k)
    a = torch.empty(k, ld, device=DEV, dtype=torch.bfloat16)[:, ld - 64:]
    a.copy_(torch.randn(k, 64, generator=g, device=DEV))
    b = torch.randn(k, 72, generator=g, device=DEV).bfloat16()
    c = host().product(a, True, b, True, 0, None)
    ref = a.double().t().contiguous() @ b.double()
    bound = (k + 4) * 2.0 ** -24 * (a.double().abs().t().contiguous() @ b.double().abs()) + 2.0 ** -8 * ref.abs()
    assert torch.all((c.double() - ref).abs() <= 1.01 * bound)


def test_projection_of_rows_beyond_32_bit_offsets():
    """Rows that lie further apart than the products' offsets reach: 40000 of them, 65536 elements apart."""
    from lookahead_keys_attention_amd import Castle

    torch.manual_seed(0)
    model = Castle(64, heads=1, dim_head=16, use_triton=True).to(DEV).bfloat16()
    wide = torch.empty(8, 5000, 65536, device=DEV, dtype=torch.bfloat16)
    x = wide[..., :64]
    x.copy_(torch.randn(8, 5000, 64, device=DEV))
    with pytest.raises(ValueError):
        host().product(x.flatten(0, 1), False, model.to_all_qkv.weight.detach(), False, 0, None)
    results = []
    for rows in (x, x.contiguous()):
        leaf = rows.detach().requires_grad_()
        y = model(leaf)
        results.append([y, *torch.autograd.grad(y.float().square().sum(), [leaf, *model.parameters()])])
    for a, b in zip(*results):   # (the library's products and the kernels' order their sums differently)
        assert (a - b).float().norm() <= 1e-2 * b.float().norm()


def test_rows_that_overlap_in_memory():
    """Inputs and output gradients whose rows are one row repeated (stride 0), or windows of one row: a sum over the
    sequence hands such gradients back."""
    from lookahead_keys_attention_amd import Castle

    torch.manual_seed(0)
    line = torch.randn(1, 1, 64 + 8 * 39, device=DEV)
    for prenorm in (False, True):
        model = Castle(64, heads=2, dim_head=32, use_triton=True, prenorm=prenorm).to(DEV)
        for x in (line[..., :64].expand(2, 40, 64), line[0].unfold(1, 64, 8), torch.randn(1, 40, 64, device=DEV)):
            for pool in (lambda y: y.sum(dim=1), lambda y: y.sum(dim=(0, 1))):
                results = []
                for rows in (x, x.contiguous()):
                    y = model(rows)
                    pooled = pool(y) if rows is x else pool(y * 1)   # (the product's gradient is contiguous)
                    results.append([y, *torch.autograd.grad(pooled.square().sum(), model.parameters())])
                for a, b in zip(*results):   # (other products, so other orders of the 32-bit sums)
                    assert (a - b).norm() <= 1e-4 * b.norm()


@pytest.mark.parametrize("rows,n,k,column,columns", [(1, 64, 64, 8, 16), (130, 576, 128, 192, 96), (1000, 1536, 256, 512, 256), (2048, 512, 256, 0, 512),
                                                     (5000, 3072, 512, 1024, 512)])
def test_product_leaves_partial_maxima(rows, n, k, column, columns):
    """The largest element of some columns, taken on the store: column ranges inside, across and at the ends of tiles."""
    import ctypes

    from lookahead_keys_attention_amd import _native as N

    class Amax(ctypes.Structure):
        _fields_ = [("partials", ctypes.c_void_p), ("status", ctypes.c_void_p), ("column", ctypes.c_int32), ("columns", ctypes.c_int32)]

    lib = N.lib()
    vp, i, i64 = ctypes.c_void_p, ctypes.c_int, ctypes.c_int64
    lib.castle_gemm.argtypes = [vp, i64, i, vp, i64, i, vp, i64, i, i, i, i, i, vp, ctypes.POINTER(Amax), vp, i64, vp]
    assert lib.castle_gemm_amax_ok(rows, n, k, 1, column, columns)
    g = torch.Generator(device=DEV).manual_seed(rows)
    x, w = (torch.randn(*s, generator=g, device=DEV).bfloat16() for s in ((rows, k), (n, k)))
    c, part = torch.empty(rows, n, device=DEV, dtype=torch.bfloat16), torch.full((257,), -1.0, device=DEV)
    for r, col in ((0, column), (rows - 1, column + columns - 1), (rows // 2, column + columns // 2)):
        w[col] += 3 * x[r] / x[r].norm() * k ** 0.5   # the largest element sits there, and one just outside must not count
        if column > 0:
            w[column - 1] += 9 * x[r]
        amax = Amax(part.data_ptr(), part[256:].data_ptr(), column, columns)
        N.check(lib.castle_gemm(x.data_ptr(), k, 0, w.data_ptr(), k, 0, c.data_ptr(), n, rows, n, k, 1, 0, None, ctypes.byref(amax), None, 0,
                                N.stream_ptr(x.device)), "castle_gemm")
        torch.cuda.synchronize()
        assert part[:256].max() == c[:, column:column + columns].float().abs().max() and part[:256].min() >= 0 and part[256:].view(torch.int32).item() == 0
