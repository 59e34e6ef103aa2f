"""Parity of the HIP path (through the C ABI) with the CPU oracle, on the GPU.

Tolerances (binding, from the north star and the reference's own tests):
  fp32 : outputs max|a-b| <= 1e-3, gradients <= 2e-2        (tests/test_lookahead.py:114,135 of the reference)
  bf16 : against the oracle evaluated in fp64 on the same bf16-rounded inputs,
         max|a-b| <= 2e-2 * max|b|  and  ||a-b|| <= 2e-2 * ||b||
"""
import pytest
import torch

pytestmark = pytest.mark.gpu

from oracle import castle_oracle as O

DEV = "cuda:0"
NAMES = ("dqc", "dkc", "dvc", "dqu", "dku", "dvu")


def H():
    from lookahead_keys_attention_amd import ops

    return ops


def rand_ops(B, Hh, L, d, dtype, seed, scale=0.6):
    g = torch.Generator().manual_seed(seed)
    ops = [(torch.randn(B, Hh, L, d, generator=g) * scale).to(dtype) for _ in range(6)]
    dout = torch.randn(B, Hh, L, d, generator=g).to(dtype)
    return ops, dout


def assert_close(got, ref, dtype, what, fp32_atol):
    got, ref = got.detach().cpu().double(), ref.double()
    err = (got - ref).abs().max().item()
    if dtype == torch.float32:
        assert err <= fp32_atol, f"{what}: max err {err:.3e} > {fp32_atol}"
    else:
        assert err <= 2e-2 * ref.abs().max().item(), f"{what}: max err {err:.3e} vs max {ref.abs().max():.3e}"
        rel = ((got - ref).norm() / ref.norm()).item()
        assert rel <= 2e-2, f"{what}: relative norm error {rel:.3e}"


FWD_CASES = [
    (1, 1, 1, 64, torch.float32), (1, 2, 7, 16, torch.float32), (2, 2, 64, 64, torch.float32),
    (1, 2, 65, 32, torch.float32), (2, 2, 200, 32, torch.float32), (1, 2, 257, 64, torch.float32),
    (1, 1, 384, 16, torch.float32), (2, 2, 384, 64, torch.bfloat16), (1, 2, 300, 128, torch.bfloat16),
    (1, 2, 130, 32, torch.bfloat16), (1, 2, 256, 64, torch.float16),
]


@pytest.mark.parametrize("B,Hh,L,d,dtype", FWD_CASES)
def test_operator_forward(B, Hh, L, d, dtype):
    ops, _ = rand_ops(B, Hh, L, d, dtype, seed=L + d)
    s = d ** -0.5
    out, U = H().castle_attention_hip(*[t.to(DEV) for t in ops], s, True)
    ref_out, ref_U = O.parallel_core(*[t.double() for t in ops], s, want_U=True)
    assert out.shape == (B, Hh, L, d) and U.shape == (B, Hh, L, d) and out.dtype == dtype
    assert_close(out, ref_out, dtype, "out", 1e-3)
    if L > 1:
        assert_close(U, ref_U, dtype, "U", 1e-3)
    assert torch.all(U[:, :, -1] == 0)


BWD_CASES = [
    (1, 1, 1, 64, torch.float32), (1, 2, 9, 16, torch.float32), (2, 2, 64, 64, torch.float32),
    (1, 2, 200, 32, torch.float32), (1, 2, 321, 64, torch.float32), (2, 2, 384, 64, torch.bfloat16),
    (1, 2, 300, 32, torch.bfloat16), (1, 2, 256, 16, torch.bfloat16), (1, 2, 256, 64, torch.float16),
    (1, 2, 300, 128, torch.bfloat16), (1, 1, 130, 128, torch.float16),
    (1, 3, 129, 16, torch.bfloat16), (3, 1, 448, 64, torch.float16), (1, 9, 640, 64, torch.bfloat16),
    (2, 3, 709, 128, torch.bfloat16),
]


@pytest.mark.parametrize("B,Hh,L,d,dtype", BWD_CASES)
def test_operator_backward(B, Hh, L, d, dtype):
    ops, dout = rand_ops(B, Hh, L, d, dtype, seed=3 * L + d)
    s = d ** -0.5
    leaves = [t.to(DEV).requires_grad_() for t in ops]
    H().castle_attention_hip(*leaves, s).backward(dout.to(DEV))
    ref = O.closed_form_grads(*[t.double() for t in ops], s, dout.double())
    for name, leaf, r in zip(NAMES, leaves, ref):
        assert_close(leaf.grad, r, dtype, name, 2e-2)
        if dtype == torch.float32:      # far inside the bound in practice
            assert (leaf.grad.cpu().double() - r).abs().max() <= 1e-4, name


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("B,Hh,L,d", [(2, 3, 5, 64), (1, 2, 31, 32), (2, 2, 33, 64), (1, 3, 65, 16), (2, 2, 95, 128), (1, 2, 97, 64), (1, 1, 545, 128),
                                      (1, 2, 800, 32), (10, 52, 5, 64), (8, 66, 33, 32), (10, 52, 64, 64), (8, 66, 97, 64), (4, 130, 129, 16), (4, 65, 130, 128)])
def test_operator_at_tile_edges_with_few_and_with_many_heads(B, Hh, L, d, dtype):
    """Few heads take the kernels over 32-row items, many (more than two workgroups of 128 rows per CU) those over 128."""
    if dtype == torch.float32 and d == 128:
        pytest.skip("no fp32 kernels at d = 128")
    ops, dout = rand_ops(B, Hh, L, d, dtype, seed=5 * L + d)
    s = d ** -0.5
    leaves = [t.to(DEV).requires_grad_() for t in ops]
    out, U = H().castle_attention_hip(*leaves, s, True)
    out.backward(dout.to(DEV))
    ref_out, ref_U = O.parallel_core(*[t.double() for t in ops], s, want_U=True)
    assert_close(out, ref_out, dtype, "out", 1e-4)
    assert_close(U, ref_U, dtype, "U", 1e-4)
    for name, leaf, r in zip(NAMES, leaves, O.closed_form_grads(*[t.double() for t in ops], s, dout.double())):
        assert_close(leaf.grad, r, dtype, name, 1e-4)


@pytest.mark.parametrize("B,Hh,L,d", [(1, 1, 481, 64), (1, 1, 513, 64), (2, 3, 545, 32), (1, 5, 1024, 16), (1, 9, 1025, 64), (1, 1, 2049, 64)])
def test_operator_with_long_walks_shared_by_eight_waves(B, Hh, L, d):
    """Few heads of many rows, at both ends of the range of that choice and with segments of unequal length."""
    test_operator_at_tile_edges_with_few_and_with_many_heads(B, Hh, L, d, torch.bfloat16)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("Hh,L", [(300, 1), (257, 33), (512, 96), (257, 128), (130, 129), (100, 352), (40, 1000), (65, 385), (96, 500), (60, 705), (33, 961), (33, 993), (64, 1024)])
def test_wide_heads_by_two_groups_of_waves(Hh, L, dtype):
    """d = 128 at one and two row blocks a CU, where two groups of waves share the keys of a row if a head has four row blocks or more, against the same heads
    among others: odd and even numbers of chunks, a last one that only the first group has."""
    g = torch.Generator(device="cuda").manual_seed(L)
    six = [torch.randn(1, Hh, L, 128, generator=g, device="cuda").to(dtype) for _ in range(6)]
    blocks = Hh * ((L + 127) // 128)
    assert 256 < blocks <= 512
    few = H().castle_attention_hip(*six, 128 ** -0.5)
    many = H().castle_attention_hip(*(t.repeat(512 // blocks + 1, 1, 1, 1) for t in six), 128 ** -0.5)
    # both round their sums of at most the largest value, of weights rounded to fp16 behind maxima of their own
    bits = 8 if dtype == torch.bfloat16 else 11
    bound = 2.0 ** -(bits - 1) * many[0].float().abs() + 2.0 ** -9 * six[2].float().abs().max()
    assert torch.isfinite(few).all() and torch.all((few[0].float() - many[0].float()).abs() <= bound)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("first,last", [(32, 128), (0, 64), (64, 320)])
def test_wide_heads_with_scores_of_minus_infinity(first, last, dtype):
    """Keys whose scores are -inf have no weight, also where one of two groups of waves sees nothing else at first: what many heads, by one group, and
    the oracle give without them."""
    Hh, L, d = 65, 480, 128
    g = torch.Generator(device="cuda").manual_seed(first)
    six = [torch.randn(1, Hh, L, d, generator=g, device="cuda").to(dtype) for _ in range(6)]
    six[0][..., 0] = six[0][..., 0].abs() + 0.1
    six[1][:, :, first:last, 0] = float("-inf")
    few = H().castle_attention_hip(*six, d ** -0.5)
    many = H().castle_attention_hip(*(t.repeat(2, 1, 1, 1) for t in six), d ** -0.5)[:1]
    seen = slice(last if first == 0 else 0, L)   # (a row that sees no other key has no result)
    ref = O.parallel_core(*[t[:, :1].cpu().double() for t in six], d ** -0.5, want_U=False)
    ref = ref[0] if isinstance(ref, tuple) else ref
    for out in (few, many):
        assert torch.isfinite(out[:, :, seen]).all()
        if first == 0 and dtype is torch.float16:   # (bf16 rows are saturated on their way to fp16)
            assert out[:, :, :last].isnan().all()
        assert_close(out[:, :1, seen], ref[:, :, seen], dtype, "out", 1e-3)


@pytest.mark.parametrize("L,d", [(256, 64), (200, 32)])
def test_bf16_operand_flag_forward_and_backward(L, d, monkeypatch):
    """CASTLE_FLAG_BF16_OPERANDS keeps bf16 MFMA operands (default: fp16 operands for bf16 tensors)."""
    from lookahead_keys_attention_amd import _native

    monkeypatch.setattr(H(), "DEFAULT_FLAGS", _native.FLAG_BF16_OPERANDS)
    ops, dout = rand_ops(2, 2, L, d, torch.bfloat16, seed=L + 7 * d)
    s = d ** -0.5
    leaves = [t.to(DEV).requires_grad_() for t in ops]
    out, U = H().castle_attention_hip(*leaves, s, True)
    out.backward(dout.to(DEV))
    ref_out, ref_U = O.parallel_core(*[t.double() for t in ops], s, want_U=True)
    assert_close(out, ref_out, torch.bfloat16, "out", 1e-3)
    assert_close(U, ref_U, torch.bfloat16, "U", 1e-3)
    ref = O.closed_form_grads(*[t.double() for t in ops], s, dout.double())
    for name, leaf, r in zip(NAMES, leaves, ref):
        assert_close(leaf.grad, r, torch.bfloat16, name, 2e-2)


@pytest.mark.parametrize("B,Hh,L,d,dtype", [(1, 2, 200, 64, torch.float32), (2, 2, 300, 64, torch.bfloat16),
                                            (1, 2, 130, 32, torch.float16), (1, 1, 260, 128, torch.bfloat16)])
def test_rotary_inside_the_kernels(B, Hh, L, d, dtype):
    """FLAG_ROTARY: rotating inside the kernels == the operator on operands rotated beforehand by
    the oracle's rotary embedding (complex multiplication, fp64), forward, final lookahead keys and
    the gradients with respect to the UN-rotated operands (chain rule through the rotation)."""
    ops, dout = rand_ops(B, Hh, L, d, dtype, seed=5 * L + d)
    s = d ** -0.5
    leaves = [t.to(DEV).requires_grad_() for t in ops]
    out, U = H().castle_attention_hip(*leaves, s, True, rotary=True)
    out.backward(dout.to(DEV))
    pos = torch.arange(L)
    rot = [t.double() if idx == 2 else O.rope(t.double(), pos) for idx, t in enumerate(ops)]
    ref_out, ref_U = O.parallel_core(*rot, s, want_U=True)
    assert_close(out, ref_out, dtype, "out", 1e-3)
    assert_close(U, ref_U, dtype, "U", 1e-3)
    # gradients: closed forms with respect to the rotated operands, rotated back (transpose = -angle)
    g_rot = O.closed_form_grads(*rot, s, dout.double())
    inv = lambda g: O.rope(g, -pos)
    for idx, (name, leaf) in enumerate(zip(NAMES, leaves)):
        want = g_rot[idx] if idx == 2 else inv(g_rot[idx])
        assert_close(leaf.grad, want, dtype, name, 2e-2)


def test_rope_entry_point_matches_formula():
    x = torch.randn(2, 3, 77, 64, generator=torch.Generator().manual_seed(2))
    for dtype, tol in ((torch.float32, 1e-4), (torch.bfloat16, 2e-2)):
        xs = x.to(dtype).to(DEV)
        out = torch.empty_like(xs)
        H().castle_rope_hip(xs, out, first_position=11)
        want = O.rope(x.to(dtype).double(), torch.arange(11, 11 + 77))
        assert (out.double().cpu() - want).abs().max() <= tol


@pytest.mark.parametrize("d", [64, 128])
def test_backward_without_score_tiles(d, monkeypatch):
    """Long sequences do not get the dS / dSu tile buffers (they grow with L^2); the second backward
    kernel then recomputes the score chain (at d = 128 both single-role kernels run, in two passes
    each).  Forced here through FLAG_RECOMPUTE_SCORES."""
    from lookahead_keys_attention_amd import _native

    small = _native.lib().castle_bwd_workspace_bytes(2, 2, 300, d, 1, _native.FLAG_RECOMPUTE_SCORES)
    assert small < _native.lib().castle_bwd_workspace_bytes(2, 2, 300, d, 1, 0)
    monkeypatch.setattr(H(), "DEFAULT_FLAGS", _native.FLAG_RECOMPUTE_SCORES)
    ops, dout = rand_ops(2, 2, 300, d, torch.bfloat16, seed=77)
    s = d ** -0.5
    leaves = [t.to(DEV).requires_grad_() for t in ops]
    H().castle_attention_hip(*leaves, s).backward(dout.to(DEV))
    ref = O.closed_form_grads(*[t.double() for t in ops], s, dout.double())
    for name, leaf, r in zip(NAMES, leaves, ref):
        assert_close(leaf.grad, r, torch.bfloat16, name, 2e-2)


def test_gradients_are_linear_in_the_upstream_gradient_down_to_tiny_magnitudes():
    """The backward runs on dO times a power of two chosen from max|dO| (16-bit operands), so a tiny
    or a huge upstream gradient gives EXACTLY the scaled gradients of an ordinary one: nothing is
    flushed to zero on the way through the fp16 dS / dSu / dZ operands (a mean-reduced loss over 16k
    tokens hands down |dO| ~ 1e-5).  Powers of two, so the comparison is bit for bit."""
    ops, dout = rand_ops(1, 2, 384, 64, torch.bfloat16, seed=21)
    s = 64 ** -0.5

    def grads(factor):
        leaves = [t.to(DEV).requires_grad_() for t in ops]
        H().castle_attention_hip(*leaves, s).backward((dout * factor).to(DEV))
        return [leaf.grad.float().cpu() for leaf in leaves]

    base = grads(1.0)
    ref = O.closed_form_grads(*[t.double() for t in ops], s, dout.double())
    for name, got, r in zip(NAMES, base, ref):
        assert_close(got, r, torch.bfloat16, name, 2e-2)
    for k in (-24, -12, 12):
        scaled = grads(2.0 ** k)
        for name, a, b in zip(NAMES, scaled, base):
            assert torch.equal(a * 2.0 ** -k, b), f"{name} at dout * 2^{k}"


@pytest.mark.parametrize("L,vu_gain,vu_mean,q_gain,grads_in_tolerance",
                         [(512, 10.0, 0.0, 1.0, True), (1024, 300.0, 150.0, 0.25, False), (640, 4000.0, 2000.0, 0.02, False)])
def test_large_lookahead_states_stay_inside_the_fp16_range(L, vu_gain, vu_mean, q_gain, grads_in_tolerance):
    """Lookahead states far larger than unit-variance operands give.  vu is pre-scaled by a power of
    two chosen on the device from max|vu| (L * max|vu_s| <= 2^15), so no state overflows the fp16
    operands however large vu is: U stays within the bf16 tolerance, the output within it normwise,
    and every gradient is finite (|U| up to 7.5e5 here).  Precision is another matter: the fp16 operands carry 11 bits, so
    Su = qc . U is known to about 2^-11 |qc| |U|; with |Su| ten times the default-init regime
    (|U| ~ 200, |Su| ~ 150, first case) all gradients are still inside the tolerance, beyond that
    the gradients that pass through silu'(Su) (dqc, dqu, dku, dvu) lose accuracy and only dkc, dvc
    are held to a bound."""
    ops, dout = rand_ops(1, 2, L, 64, torch.bfloat16, seed=L)
    ops[5] = (ops[5].float() * vu_gain + vu_mean).bfloat16()   # a mean makes U grow like L
    ops[0] = (ops[0].float() * q_gain).bfloat16()
    s = 64 ** -0.5
    leaves = [t.to(DEV).requires_grad_() for t in ops]
    out, U = H().castle_attention_hip(*leaves, s, True)
    out.backward(dout.to(DEV))
    ref_out, ref_U = O.parallel_core(*[t.double() for t in ops], s, want_U=True)
    assert ref_U.abs().max() > 200
    assert torch.isfinite(out).all() and torch.isfinite(U).all()
    rel_norm = lambda got, want: ((got.detach().cpu().double() - want).norm() / want.norm()).item()
    assert_close(U, ref_U, torch.bfloat16, "U", 1e-3)
    if grads_in_tolerance:
        assert_close(out, ref_out, torch.bfloat16, "out", 1e-3)
    else:
        assert rel_norm(out, ref_out) <= 2e-2
    ref = O.closed_form_grads(*[t.double() for t in ops], s, dout.double())
    for name, leaf, r in zip(NAMES, leaves, ref):
        assert torch.isfinite(leaf.grad).all(), name
        if grads_in_tolerance:
            assert_close(leaf.grad, r, torch.bfloat16, name, 2e-2)
        elif name in ("dkc", "dvc"):
            assert rel_norm(leaf.grad, r) <= 2e-2, name


def test_bf16_inputs_beyond_the_fp16_range_are_clamped_and_reported(monkeypatch):
    """A bf16 tensor can hold |x| > 65504, the fp16 operands cannot: such elements are clamped when
    the operands are copied, the kernels say so in the workspace header (ops.CHECK_RANGE turns that
    into an error), and the result is that of the clamped operands."""
    ops, _ = rand_ops(1, 2, 256, 64, torch.bfloat16, seed=31)
    ops[1][0, 0, 17, 5] = 3.0e5      # kc
    ops[2][0, 1, 40, 9] = -1.0e6     # vc
    s = 64 ** -0.5
    dev = [t.to(DEV) for t in ops]
    out = H().castle_attention_hip(*dev, s)
    assert torch.isfinite(out).all()
    clamped = [t.double().clamp(-65504.0, 65504.0) for t in ops]
    assert_close(out, O.parallel_core(*clamped, s), torch.bfloat16, "out", 1e-3)
    monkeypatch.setattr(H(), "CHECK_RANGE", True)
    with pytest.raises(RuntimeError, match="clamped"):
        H().castle_attention_hip(*dev, s)
    ops2, _ = rand_ops(1, 2, 256, 64, torch.bfloat16, seed=31)
    H().castle_attention_hip(*[t.to(DEV) for t in ops2], s)     # in range: no complaint


@pytest.mark.parametrize("L,d,dtype", [(640, 64, torch.bfloat16), (300, 32, torch.float32), (260, 128, torch.bfloat16)])
def test_backward_that_recomputes_the_forward_state(L, d, dtype, monkeypatch):
    """KEEP_STATE_LIMIT_BYTES = 0: the snapshot buffer is dropped after the forward pass (what the call
    keeps is O(L d)) and castle_bwd runs the scan again first (FLAG_RECOMPUTE_STATE).  Same kernels,
    same inputs: the gradients are bit for bit those of the run that kept the snapshots."""
    ops, dout = rand_ops(1, 2, L, d, dtype, seed=L + 1)
    s = d ** -0.5

    def grads():
        leaves = [t.to(DEV).requires_grad_() for t in ops]
        H().castle_attention_hip(*leaves, s).backward(dout.to(DEV))
        return [leaf.grad.cpu() for leaf in leaves]

    kept = grads()
    monkeypatch.setattr(H(), "KEEP_STATE_LIMIT_BYTES", 0)
    again = grads()
    for name, a, b in zip(NAMES, kept, again):
        assert torch.equal(a, b), name
    ref = O.closed_form_grads(*[t.double() for t in ops], s, dout.double())
    for name, got, r in zip(NAMES, again, ref):
        assert_close(got, r, dtype, name, 2e-2)


def test_two_streams_run_the_operator_side_by_side():
    """Every launch goes to the caller's stream and every call owns its workspace: two forward +
    backward passes enqueued on two streams without synchronising in between give, bit for bit,
    what each gives alone on the default stream."""
    cases = [(2, 2, 640, 64, torch.bfloat16, 5), (1, 4, 384, 32, torch.bfloat16, 6)]
    alone = []
    for B, Hh, L, d, dtype, seed in cases:
        ops, dout = rand_ops(B, Hh, L, d, dtype, seed=seed)
        leaves = [t.to(DEV).requires_grad_() for t in ops]
        out = H().castle_attention_hip(*leaves, d ** -0.5)
        out.backward(dout.to(DEV))
        alone.append((out.detach().clone(), [leaf.grad.clone() for leaf in leaves]))
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream(device=DEV) for _ in cases]
    together = []
    for (B, Hh, L, d, dtype, seed), stream in zip(cases, streams):
        ops, dout = rand_ops(B, Hh, L, d, dtype, seed=seed)
        leaves = [t.to(DEV).requires_grad_() for t in ops]
        dout = dout.to(DEV)
        torch.cuda.synchronize()
        together.append((leaves, dout, stream))
    results = []
    for leaves, dout, stream in together:      # enqueue both before waiting for either
        with torch.cuda.stream(stream):
            out = H().castle_attention_hip(*leaves, leaves[0].shape[-1] ** -0.5)
            out.backward(dout)
            results.append(out)
    torch.cuda.synchronize()
    for (want_out, want_grads), out, (leaves, _, _) in zip(alone, results, together):
        assert torch.equal(out, want_out)
        for leaf, want in zip(leaves, want_grads):
            assert torch.equal(leaf.grad, want)


def test_forward_and_backward_are_deterministic():
    """No atomics anywhere: the same inputs give the same bits, call after call."""
    ops, dout = rand_ops(2, 3, 1000, 64, torch.bfloat16, seed=9)
    runs = []
    for _ in range(3):
        leaves = [t.to(DEV).requires_grad_() for t in ops]
        out = H().castle_attention_hip(*leaves, 0.125)
        out.backward(dout.to(DEV))
        runs.append([out.detach()] + [leaf.grad for leaf in leaves])
    for other in runs[1:]:
        assert all(torch.equal(a, b) for a, b in zip(runs[0], other))


def test_lookahead_keys_carry_no_gradient():
    ops, dout = rand_ops(1, 1, 40, 16, torch.float32, seed=5)
    leaves = [t.to(DEV).requires_grad_() for t in ops]
    out, U = H().castle_attention_hip(*leaves, 0.25, True)
    assert out.requires_grad and not U.requires_grad   # lookahead_keys_attention_triton.py:513-515


def test_zero_lookahead_values_equal_sdpa():
    ops, _ = rand_ops(2, 2, 150, 64, torch.float32, seed=6)
    qc, kc, vc, qu, ku, vu = [t.to(DEV) for t in ops]
    out = H().castle_attention_hip(qc, kc, vc, qu, ku, torch.zeros_like(vu), 64 ** -0.5)
    ref = torch.nn.functional.scaled_dot_product_attention(*[t.double() for t in ops[:3]], is_causal=True)
    assert (out.cpu().double() - ref).abs().max() <= 1e-4


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_packed_operator_equals_unpacked(dtype):
    B, L, heads, d = 2, 200, 2, 64
    g = torch.Generator().manual_seed(8)
    proj = (torch.randn(B, L, 6 * heads * d, generator=g) * 0.6).to(dtype).to(DEV).requires_grad_()
    dmerged = torch.randn(B, L, heads * d, generator=g).to(dtype).to(DEV)
    merged, U = H().castle_attention_packed(proj, heads, d ** -0.5, True)
    merged.backward(dmerged)
    g_packed = proj.grad.clone()
    proj.grad = None
    qu, ku, vu, qc, kc, vc = proj.view(B, L, 6, heads, d).permute(2, 0, 3, 1, 4).unbind(0)
    out2, U2 = H().castle_attention_hip(qc, kc, vc, qu, ku, vu, d ** -0.5, True)
    merged2 = out2.permute(0, 2, 1, 3).reshape(B, L, heads * d)
    merged2.backward(dmerged)
    assert torch.equal(merged, merged2) and torch.equal(U, U2)
    assert torch.equal(g_packed, proj.grad)


DEC_CASES = [(2, 2, 0, 40, 64, torch.float32), (2, 2, 100, 30, 64, torch.float32), (1, 3, 300, 20, 16, torch.float32),
             (1, 2, 70, 10, 32, torch.float32), (2, 2, 200, 20, 64, torch.bfloat16), (1, 2, 130, 10, 128, torch.bfloat16),
             # many row splits per (b, h): 24 (three batches of the merge) and the cap of 64
             (1, 2, 1500, 4, 64, torch.float32), (1, 1, 4200, 3, 32, torch.bfloat16)]


@pytest.mark.parametrize("B,Hh,t0,steps,d,dtype", DEC_CASES)
def test_decode_steps(B, Hh, t0, steps, d, dtype):
    L = t0 + steps
    ops, _ = rand_ops(B, Hh, L, d, dtype, seed=11 * L + d)
    s = d ** -0.5
    ref = [t.double() for t in ops]
    ref_out, ref_U = O.parallel_core(*ref, s, want_U=True)
    bufs = [torch.zeros(B, Hh, L + 3, d, dtype=dtype, device=DEV) for _ in range(4)]
    if t0:
        _, U0 = O.parallel_core(*[t[:, :, :t0] for t in ref], s, want_U=True)
        for buf, src in zip(bufs, (U0.to(dtype), ops[3][:, :, :t0], ops[1][:, :, :t0], ops[2][:, :, :t0])):
            buf[:, :, :t0] = src.to(DEV)
    ws = H().decode_workspace(B, Hh, d, DEV)
    dev_ops = [t.to(DEV) for t in ops]
    outs = []
    for t in range(t0, L):
        o = torch.empty(B, Hh, 1, d, dtype=dtype, device=DEV)
        H().castle_decode_step_hip(*bufs, t, *[x[:, :, t:t + 1] for x in dev_ops], s, o, ws)
        outs.append(o)
    got = torch.cat(outs, 2)
    assert_close(got, ref_out[:, :, t0:], dtype, "decode out", 1e-3)
    if dtype == torch.float32:
        assert_close(bufs[0][:, :, :L], ref_U, dtype, "U", 1e-3)
    assert torch.equal(bufs[1][:, :, :L].cpu(), ops[3]) and torch.equal(bufs[2][:, :, :L].cpu(), ops[1])
    assert torch.equal(bufs[3][:, :, :L].cpu(), ops[2])


@pytest.mark.parametrize("Hh,d,dtype,t", [(3, 64, torch.bfloat16, 0), (3, 64, torch.bfloat16, 65), (2, 16, torch.float16, 300), (2, 128, torch.float16, 47), (1, 32, torch.float32, 130)])
def test_decode_step_ignores_what_lies_beyond_the_count(Hh, d, dtype, t):
    """The whole ring is read before the row count is known: NaN in every row and ring slot that holds nothing changes no bit, with the count from the host and from the device, and caches whose strides differ give the same bits."""
    from lookahead_keys_attention_amd import _native as N
    from lookahead_keys_attention_amd.castle import _CacheStore

    B, cap = 2, t + 130
    g = torch.Generator(device=DEV).manual_seed(t + d)
    rnd = lambda *shape: (torch.randn(*shape, generator=g, device=DEV) * 0.6).to(dtype)
    rows, steps = [rnd(B, Hh, t, d) for _ in range(4)], [[rnd(B, Hh, 1, d) for _ in range(6)] for _ in range(3)]
    results = []
    for kind in ("zero", "nan", "device", "strides", "strides, read once"):
        store = _CacheStore(B, Hh, d, cap, dtype, torch.device(DEV))
        fill = 0.0 if kind == "zero" else float("nan")
        caches = [torch.full((B, Hh, cap, d + (16 * i if kind.startswith("strides") else 0)), fill, dtype=dtype, device=DEV)[..., :d] for i in range(4)]
        for cache, row in zip(caches, rows):
            cache[:, :, :t] = row
        for extra in store.rings:
            extra.fill_(fill)
        outs = []
        for i, token in enumerate(steps):
            out = torch.empty(B, Hh, 1, d, dtype=dtype, device=DEV)
            deferred = H().make_deferred(store.rings[0], store.rings[1], t)
            if kind == "device":
                count = torch.tensor([t + i], dtype=torch.int32, device=DEV)
                N.check(N.lib().castle_decode_step_device_count(*[N.view4(c) for c in caches], count.data_ptr(), cap, *[N.view4(x) for x in token], B, Hh, d,
                                                                N.dtype_code(dtype), d ** -0.5, N.FLAG_ROTARY, N.view4(out), deferred, store.workspace.data_ptr(),
                                                                store.workspace.numel(), N.stream_ptr(out.device)), "castle_decode_step_device_count")
            elif kind == "strides, read once":
                N.check(N.lib().castle_decode_step(*[N.view4(c) for c in caches], t + i, cap, *[N.view4(x) for x in token], B, Hh, d, N.dtype_code(dtype),
                                                   d ** -0.5, N.FLAG_ROTARY | N.FLAG_READ_ONCE, N.view4(out), deferred, store.workspace.data_ptr(),
                                                   store.workspace.numel(), N.stream_ptr(out.device)), "castle_decode_step")
            else:
                H().castle_decode_step_hip(*caches, t + i, *token, d ** -0.5, out, store.workspace, rotary=True, deferred=deferred)
            outs.append(out)
        results.append((torch.cat(outs, 2), torch.stack([c[:, :, :t + 3] for c in caches])))
    for out, cached in results:
        assert torch.isfinite(out.float()).all()
    for (out, cached), kind in zip(results[1:], ("nan", "device", "strides", "strides, read once")):
        if kind == "device":   # (its splits are those of a full cache: sums in another order, roundings of the results)
            assert_close(out.float(), results[0][0].cpu().double(), dtype, kind, 1e-5)
        else:
            assert torch.equal(out, results[0][0]) and torch.equal(cached, results[0][1]), kind


@pytest.mark.parametrize("M,N,K,dtype", [(32, 3072, 512, torch.bfloat16), (32, 512, 512, torch.bfloat16), (1, 96, 32, torch.float16),
                                         (5, 6 * 2 * 16, 40, torch.bfloat16), (64, 130, 264, torch.float16), (33, 64, 2048, torch.bfloat16)])
def test_small_linear_matches_fp64_matmul(M, N, K, dtype):
    """The projections around the cached step (lookahead_keys_attention.py:99, 209 with seq_len == 1):
    y = x w^T with fp32 accumulation, against the product of the same 16-bit values in fp64; ragged
    tiles, K not a multiple of the per-wave slices."""
    g = torch.Generator().manual_seed(M + N + K)
    x = torch.randn(M, 1, K, generator=g).to(dtype)
    w = (torch.randn(N, K, generator=g) * K ** -0.5).to(dtype)
    assert H().small_linear_ok(x.to(DEV), w.to(DEV))
    y = H().small_linear(x.to(DEV), w.to(DEV))
    ref = x[:, 0].double() @ w.double().t()
    assert y.shape == (M, 1, N) and y.dtype == dtype
    err = (y[:, 0].cpu().double() - ref).abs().max().item()
    assert err <= 2.0 ** (-8 if dtype == torch.bfloat16 else -11) * ref.abs().max().item() * 1.01 + 1e-6   # one rounding of the result


@pytest.mark.parametrize("M,N,K,dtype,norm,act,res", [(16, 2048, 512, torch.bfloat16, True, "gelu", False),
                                                       (16, 512, 2048, torch.bfloat16, False, None, True),
                                                       (3, 258, 264, torch.float16, True, None, True),
                                                       (33, 96, 40, torch.bfloat16, True, "gelu", True)])
def test_small_linear_with_norm_activation_and_residual(M, N, K, dtype, norm, act, res):
    """castle_small_linear_fused: RMS normalisation in front, erf GELU and a residual behind, in one
    launch, against the same chain in fp64 on the same 16-bit values (nn.RMSNorm with eps=None takes
    the machine epsilon of its 32-bit sums; the norm weight multiplies the normalised row)."""
    g = torch.Generator().manual_seed(M + N + K)
    x = (torch.randn(M, 1, K, generator=g) * 1.7).to(dtype).to(DEV)
    w = (torch.randn(N, K, generator=g) * K ** -0.5).to(dtype).to(DEV)
    r = torch.randn(M, 1, N, generator=g).to(dtype).to(DEV) if res else None
    layer = torch.nn.RMSNorm(K).to(DEV).to(dtype) if norm else None
    if norm:
        with torch.no_grad():
            layer.weight.copy_((1 + 0.3 * torch.randn(K, generator=g)).to(dtype))
    y = H().small_linear(x, w, norm=layer, activation=act, residual=r)
    ref = x.double()
    if norm:
        eps = torch.finfo(torch.float32).eps
        ref = ref * torch.rsqrt(ref.pow(2).mean(-1, keepdim=True) + eps) * layer.weight.double()
    ref = ref @ w.double().T
    if act == "gelu":
        ref = torch.nn.functional.gelu(ref)
    if res:
        ref = ref + r.double()
    assert y.shape == (M, 1, N) and y.dtype == dtype
    err = (y.double() - ref).abs().max().item()
    assert err <= 1e-2 * max(ref.abs().max().item(), 1.0), err
    # the unfused modules give the same within the rounding of their intermediate tensors
    if norm:
        mods = torch.nn.functional.linear(layer(x), w)
        if act == "gelu":
            mods = torch.nn.functional.gelu(mods)
        if res:
            mods = mods + r
        assert (y.float() - mods.float()).abs().max() <= 3e-2 * max(mods.float().abs().max().item(), 1.0)


@pytest.mark.parametrize("B,dim,Hh,d,t,dtype", [(1, 96, 1, 16, 0, torch.float32), (3, 200, 2, 32, 65, torch.bfloat16), (16, 512, 8, 64, 130, torch.float16),
                                                (17, 264, 3, 128, 33, torch.bfloat16), (33, 1100, 3, 64, 127, torch.float32)])
def test_layer_step_equals_its_parts(B, dim, Hh, d, t, dtype):
    """castle_decode_layer (norm, projection, cached step, projection, residual) against the operators around
    castle_decode_step: edges of its 16-row and 16-column tiles, ragged K, an empty cache."""
    from lookahead_keys_attention_amd.castle import _CacheStore

    g = torch.Generator(device=DEV).manual_seed(B + dim)
    rnd = lambda *shape, std=1.0: (torch.randn(*shape, generator=g, device=DEV) * std).to(dtype)
    x, norm_w = rnd(B, 1, dim), 1 + rnd(dim, std=0.2)
    w_in, w_out, res = rnd(6 * Hh * d, dim, std=dim ** -0.5), rnd(dim, Hh * d, std=(Hh * d) ** -0.5), rnd(B, 1, dim)
    stores = []
    for _ in range(2):
        store = _CacheStore(B, Hh, d, t + 9, dtype, torch.device(DEV))
        for buf in store.buffers:
            buf.zero_()
        stores.append(store)
    for i in range(4):
        rows = rnd(B, Hh, t, d, std=0.6)
        for store in stores:
            store.buffers[i][:, :, :t] = rows.to(torch.float16).view(dtype) if i == 0 and store.u_half else rows
    got = stores[0].plan.layer(x, norm_w, 1e-5, w_in, w_out, 64, t, t, d ** -0.5, True, res, None, None)
    proj = torch.nn.functional.linear(torch.nn.functional.rms_norm(x.float(), (dim,), norm_w.float(), 1e-5).to(dtype), w_in)
    core = stores[1].plan.attend(proj, t, t, d ** -0.5, True, None, None)
    want = res.float() + torch.nn.functional.linear(core.float(), w_out.float())
    assert_close(got, want.cpu().double(), dtype, "layer step", 1e-4)
    assert torch.all(stores[0].buffers[0][:, :, t] == 0)
    for a, b in zip(stores[0].buffers[1:], stores[1].buffers[1:]):
        assert_close(a[:, :, t:t + 1].float(), b[:, :, t:t + 1].float().cpu().double(), dtype, "appended row", 1e-4)


class LayerSteps:
    """castle_decode_layer_once over consecutive steps on a cache of its own: with control words (one launch) or without (three)."""

    def __init__(self, B, dim, Hh, d, dtype, rows, capacity, w_in, w_out, norm_w, once, rotary=False, deferred=True):
        import ctypes

        from lookahead_keys_attention_amd import _native as N
        from lookahead_keys_attention_amd.castle import _CacheStore

        self.lib = ctypes.CDLL(N.LIB_PATH)
        self.lib.castle_decode_layer_control_bytes.restype = ctypes.c_int64
        self.B, self.dim, self.Hh, self.d, self.dtype, self.capacity, self.deferred = B, dim, Hh, d, dtype, capacity, deferred
        self.code, self.u_half = N.DTYPE_CODES[dtype], dtype == torch.bfloat16
        self.flags = (N.FLAG_ROTARY if rotary else 0) | (N.FLAG_U_HALF if self.u_half else 0)
        self.w_in, self.w_out, self.norm_w = w_in, w_out, norm_w
        self.t0 = self.t = rows[0].shape[2]
        self.store = _CacheStore(B, Hh, d, capacity, dtype, torch.device(DEV))
        for i, row in enumerate(rows):
            self.store.buffers[i].zero_()
            self.store.buffers[i][:, :, :self.t0] = row.to(torch.float16).view(dtype) if i == 0 and self.u_half else row
        nbytes = self.lib.castle_decode_layer_control_bytes(B, Hh, d, self.code)
        self.control = torch.zeros(nbytes, dtype=torch.uint8, device=DEV) if once else None
        self.proj = torch.empty(B, 6 * Hh * d, dtype=dtype, device=DEV)

    def step(self, x, residual=None, flags=0):
        import ctypes

        from lookahead_keys_attention_amd import ops

        vp, i64, store = ctypes.c_void_p, ctypes.c_int64, self.store
        ptr = lambda t: vp(t.data_ptr() if t is not None else None)
        y = torch.empty(self.B, 1, self.dim, dtype=self.dtype, device=DEV)
        inner = self.Hh * self.d
        pending = ops.make_deferred(store.rings[0], store.rings[1], self.t0) if self.deferred else None
        rc = self.lib.castle_decode_layer_once(
            *[ctypes.byref(v) for v in store.views], self.t, None, self.capacity, ptr(x), i64(self.dim), self.dim, ptr(self.norm_w), ctypes.c_float(1e-5),
            ptr(self.w_in), i64(self.dim), ptr(self.w_out), i64(inner), ptr(residual), i64(self.dim), ptr(y), i64(self.dim), ptr(self.proj), self.B, self.Hh,
            self.d, self.code, ctypes.c_float(self.d ** -0.5), self.flags | flags, ctypes.byref(pending) if pending is not None else None, ptr(store.workspace),
            i64(store.workspace.numel()), ptr(self.control), i64(self.control.numel() if self.control is not None else 0),
            vp(torch.cuda.current_stream().cuda_stream))
        assert rc == 0
        self.t += 1
        return y


@pytest.mark.parametrize("t", [1, 40, 96, 300])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_layer_step_in_one_launch_passes_nan_on(dtype, t):
    """A token of NaN makes this and every later output of its sequence NaN, with one split and with several, as in three launches: the partial
    results of splits whose scores are all NaN count.  The other sequence stays finite."""
    B, dim, Hh, d, steps = 2, 128, 2, 64, 7
    g = torch.Generator(device=DEV).manual_seed(t)
    rnd = lambda *shape, std=1.0: (torch.randn(*shape, generator=g, device=DEV) * std).to(dtype)
    rows, w_in, w_out = [rnd(B, Hh, t, d, std=0.6) for _ in range(4)], rnd(6 * Hh * d, dim, std=dim ** -0.5), rnd(dim, Hh * d, std=(Hh * d) ** -0.5)
    one, three = (LayerSteps(B, dim, Hh, d, dtype, rows, t + steps, w_in, w_out, None, once) for once in (True, False))
    assert one.lib.castle_decode_layer_once_ok(B, Hh, d, one.code, t + steps, dim)
    for step in range(steps):
        x = rnd(B, 1, dim)
        if step == 1:
            x[0] = float("nan")
        a, b = one.step(x), three.step(x)
        assert torch.equal(a.isnan(), b.isnan()), step
        assert a[0].isnan().all() == (step >= 1) and a[1].isfinite().all(), step
        assert_close(a[1], b[1].cpu(), dtype, "the other sequence", 1e-4)


@pytest.mark.parametrize("t", [1, 40, 300])
def test_layer_step_with_a_score_of_minus_infinity(t):
    """A token whose own score overflows to -inf has no weight among the others, whichever workgroup adds it; cached rows whose scores do have none either."""
    B, dim, Hh, d = 1, 64, 2, 16
    dtype, inner = torch.float32, 2 * 16
    g = torch.Generator(device=DEV).manual_seed(t)
    rnd = lambda *shape, std=1.0: torch.randn(*shape, generator=g, device=DEV) * std
    rows, w_in, w_out = [rnd(B, Hh, t, d, std=0.6) for _ in range(4)], rnd(6 * inner, dim, std=dim ** -0.5), rnd(dim, inner, std=inner ** -0.5)
    w_in[:, 0] = 0
    w_in[3 * inner:4 * inner, 0], w_in[4 * inner:5 * inner, 0] = -1e20, 1e20   # qc and kc of a token whose first element is one
    for low in (False, True):
        if low and t > 1:   # every other cached row too: -1e20 times 1e20
            rows[2][:, :, ::2] = 1e20
        one, three = (LayerSteps(B, dim, Hh, d, dtype, rows, t + 2, w_in, w_out, None, once) for once in (True, False))
        assert one.lib.castle_decode_layer_once_ok(B, Hh, d, one.code, t, dim)
        x = rnd(B, 1, dim)
        x[:, :, 0] = 1
        a, b = one.step(x), three.step(x)
        # the largest finite score has all the weight: scores lie 1e19 apart
        proj = torch.nn.functional.linear(x.double(), w_in.double())[0, 0].view(6, Hh, d)
        gate = torch.sigmoid(rows[1][0].double() @ proj[1].unsqueeze(-1) * d ** -0.5)
        su = ((rows[0][0].double() + gate * proj[2].unsqueeze(1)) @ proj[3].unsqueeze(-1))[..., 0] * d ** -0.5
        score = (rows[2][0].double() @ proj[3].unsqueeze(-1))[..., 0] * d ** -0.5 - su * torch.sigmoid(su)
        value = torch.stack([rows[3][0, h, score[h].argmax()] for h in range(Hh)]).double()
        want = (value.reshape(-1) @ w_out.double().t()).cpu()
        for y in (a, b):
            assert_close(y[0, 0], want, dtype, "layer step", 1e-4)


@pytest.mark.parametrize("deferred", [True, False])
@pytest.mark.parametrize("B,dim,Hh,d,t0,dtype,rotary,once", [
    (1, 96, 1, 16, 0, torch.float32, True, True), (2, 512, 3, 64, 30, torch.bfloat16, True, True), (3, 200, 2, 32, 189, torch.float16, False, True),
    (17, 264, 2, 64, 94, torch.bfloat16, False, True), (1, 136, 2, 128, 93, torch.bfloat16, True, True), (2, 256, 2, 64, 700, torch.float32, False, True), (1, 256, 2, 64, 1520, torch.float32, True, True),
    (1, 136, 1, 128, 1100, torch.bfloat16, True, True), (1, 512, 1, 128, 1527, torch.float16, False, True),
    (2, 1100, 2, 64, 700, torch.float32, False, False), (1, 520, 2, 64, 30, torch.bfloat16, False, False)])
def test_layer_step_in_one_launch_equals_three(B, dim, Hh, d, t0, dtype, rotary, once, deferred):
    """castle_decode_layer_once with its control words against the same without over consecutive steps on caches of their own: around
    whole iterations of a split (32 rows at d = 64 and 16 bit, three to a split), up to 33 splits, and with the write-back every fourth step or in each.  Both
    round the projection and the attention output to the tensor type, so what differs is the order of 32-bit sums; a value of a 16-bit
    tensor in between may then round the other way: two roundings of 2^-8 (bf16) through the output projection and the store.  Only three
    launches leave the projection in the scratch."""
    steps = 9
    g = torch.Generator(device=DEV).manual_seed(B + dim)
    rnd = lambda *shape, std=1.0: (torch.randn(*shape, generator=g, device=DEV) * std).to(dtype)
    norm_w, res = 1 + rnd(dim, std=0.2), rnd(B, 1, dim)
    w_in, w_out = rnd(6 * Hh * d, dim, std=dim ** -0.5), rnd(dim, Hh * d, std=(Hh * d) ** -0.5)
    rows = [rnd(B, Hh, t0, d, std=0.6) for _ in range(4)]
    one, three = (LayerSteps(B, dim, Hh, d, dtype, rows, t0 + steps, w_in, w_out, norm_w, words, rotary, deferred) for words in (True, False))
    for step in range(steps):
        assert one.lib.castle_decode_layer_once_ok(B, Hh, d, one.code, t0 + step, dim) == once
        x = rnd(B, 1, dim)
        for steps_of in (one, three):
            steps_of.proj.fill_(7)
        ys = [steps_of.step(x, res).double() for steps_of in (one, three)]
        assert torch.all(one.proj == 7) == once and not torch.all(three.proj == 7)
        scale = ys[1].abs().max().item()
        assert (ys[0] - ys[1]).abs().max().item() <= scale * {torch.float32: 1e-4, torch.float16: 2e-3, torch.bfloat16: 1.6e-2}[dtype], step
    stores = (one.store, three.store)
    for a, b in zip(stores[0].buffers[1:], stores[1].buffers[1:]):
        assert_close(a.float(), b.float().cpu().double(), dtype, "cached rows", 1e-4)
    if one.u_half:
        a, b = (store.buffers[0].view(torch.float16).float() for store in stores)
    else:
        a, b = (store.buffers[0].float() for store in stores)
    assert_close(a, b.cpu().double(), dtype, "lookahead keys", 1e-4)


@pytest.mark.parametrize("B,dim,Hh,d,t0,dtype", [(1, 96, 1, 16, 0, torch.float32), (1, 512, 8, 64, 300, torch.bfloat16), (16, 512, 4, 64, 300, torch.bfloat16),
                                                 (17, 264, 2, 64, 94, torch.float16), (1, 136, 1, 128, 1100, torch.bfloat16), (1, 256, 2, 64, 1520, torch.float32)])
def test_layer_step_of_jobs_that_are_taken_over(B, dim, Hh, d, t0, dtype):
    """Jobs in reverse order and next to no patience: workgroups do what they had waited for, and the step comes out with the same bits.  (That they wait in vain
    in this order is what the next test sees.)"""
    from lookahead_keys_attention_amd import _native as N

    steps = 9
    g = torch.Generator(device=DEV).manual_seed(B + dim)
    rnd = lambda *shape, std=1.0: (torch.randn(*shape, generator=g, device=DEV) * std).to(dtype)
    norm_w, w_in, w_out = 1 + rnd(dim, std=0.2), rnd(6 * Hh * d, dim, std=dim ** -0.5), rnd(dim, Hh * d, std=(Hh * d) ** -0.5)
    rows = [rnd(B, Hh, t0, d, std=0.6) for _ in range(4)]
    plain, taken = (LayerSteps(B, dim, Hh, d, dtype, rows, t0 + steps, w_in, w_out, norm_w, True, True) for _ in range(2))
    for step in range(steps):
        x = rnd(B, 1, dim)
        taken.proj.fill_(7)
        ys = plain.step(x), taken.step(x, flags=N.FLAG_STEP_TAKE_OVER)
        assert torch.all(taken.proj == 7) and torch.isfinite(ys[0]).all() and torch.equal(*ys), step
    for a, b in zip(plain.store.buffers, taken.store.buffers):
        assert torch.equal(a[:, :, :t0 + steps].view(torch.uint8), b[:, :, :t0 + steps].view(torch.uint8))


@pytest.mark.parametrize("B,dim,Hh,d,t0,dtype", [(2, 96, 1, 16, 0, torch.float32), (1, 512, 8, 64, 300, torch.bfloat16), (16, 512, 4, 64, 300, torch.bfloat16),
                                                 (17, 264, 2, 64, 94, torch.float16), (3, 136, 1, 128, 200, torch.bfloat16)])
def test_layer_step_that_is_given_up_does_not_pass_for_a_good_one(B, dim, Hh, d, t0, dtype):
    """Workgroups that leave instead of taking over what they wait for: what is not there is NaN, in this step's output and, where the cache is not
    complete, in every later one.  The control words serve the next step as before."""
    from lookahead_keys_attention_amd import _native as N

    g = torch.Generator(device=DEV).manual_seed(B + dim)
    rnd = lambda *shape, std=1.0: (torch.randn(*shape, generator=g, device=DEV) * std).to(dtype)
    w_in, w_out = rnd(6 * Hh * d, dim, std=dim ** -0.5), rnd(dim, Hh * d, std=(Hh * d) ** -0.5)
    rows = [rnd(B, Hh, t0, d, std=0.6) for _ in range(4)]
    good, bad, after = (LayerSteps(B, dim, Hh, d, dtype, rows, t0 + 6, w_in, w_out, None, True) for _ in range(3))
    x = [rnd(B, 1, dim) for _ in range(6)]
    want, got = good.step(x[0]), bad.step(x[0], flags=N.FLAG_STEP_GIVE_UP)
    assert got.isnan().any() and torch.isfinite(want).all()
    assert torch.all(got.isnan() | (got == want))
    lost = bad.store.buffers[3][:, :, :t0 + 1].isnan().flatten(1).any(1)   # sequences
    for token in x[1:]:
        want, got = good.step(token), bad.step(token)
        assert got[lost].isnan().all() and torch.equal(got[~lost], want[~lost])
    after.control = bad.control
    fresh = LayerSteps(B, dim, Hh, d, dtype, rows, t0 + 6, w_in, w_out, None, True)
    for token in x:
        assert torch.equal(after.step(token), fresh.step(token))


@pytest.mark.parametrize("B,Hh,t0,steps,d,dtype,rotary", [(2, 2, 0, 23, 64, torch.float32, False), (1, 2, 101, 18, 32, torch.float32, True),
                                                        (2, 2, 203, 21, 64, torch.bfloat16, False), (1, 2, 130, 9, 128, torch.bfloat16, True)])
def test_decode_with_deferred_write_back(B, Hh, t0, steps, d, dtype, rotary):
    """castle_deferred: the lookahead keys are written on every 4th step only, the tokens in between
    are kept as pending vu rows plus their per-row gates and applied on the fly.  Every step's output equals the
    oracle's; after castle_decode_flush the stored U is the oracle's; the steps in between leave U
    untouched (that is where the traffic is saved); and at a step that does write, the U rows equal
    what the step-by-step mode holds."""
    from lookahead_keys_attention_amd import _native as N

    L = t0 + steps
    ops, _ = rand_ops(B, Hh, L, d, dtype, seed=7 * L + d)
    s = d ** -0.5
    pos = torch.arange(L)
    ref = [t.double() if (idx == 2 or not rotary) else O.rope(t.double(), pos) for idx, t in enumerate(ops)]
    ref_out, ref_U = O.parallel_core(*ref, s, want_U=True)

    def fresh():
        bufs = [torch.zeros(B, Hh, L + 3, d, dtype=dtype, device=DEV) for _ in range(4)]
        if t0:
            _, U0 = O.parallel_core(*[t[:, :, :t0] for t in ref], s, want_U=True)
            for buf, src in zip(bufs, (U0, ref[3][:, :, :t0], ref[1][:, :, :t0], ref[2][:, :, :t0])):
                buf[:, :, :t0] = src.to(dtype).to(DEV)
        return bufs

    bufs, plain = fresh(), fresh()
    rings = [torch.zeros(B, Hh, N.DECODE_DEFER, d, dtype=dtype, device=DEV),
             torch.zeros(B, Hh, L + 3, N.DECODE_DEFER, dtype=torch.float32, device=DEV)]
    ws = H().decode_workspace(B, Hh, d, DEV)
    dev_ops = [t.to(DEV) for t in ops]
    outs, wrote = [], 0
    for t in range(t0, L):
        tok = [x[:, :, t:t + 1] for x in dev_ops]
        before = bufs[0][:, :, :t].clone()
        o = torch.empty(B, Hh, 1, d, dtype=dtype, device=DEV)
        H().castle_decode_step_hip(*bufs, t, *tok, s, o, ws, rotary=rotary, deferred=H().make_deferred(*rings, t0))
        H().castle_decode_step_hip(*plain, t, *tok, s, torch.empty_like(o), ws, rotary=rotary)
        outs.append(o)
        if (t + 1) % N.DECODE_DEFER == 0:
            wrote += 1
            if dtype == torch.float32:
                assert_close(bufs[0][:, :, :t + 1], plain[0][:, :, :t + 1].cpu(), dtype, f"U at writing step {t}", 1e-5)
        elif t > 0:
            assert torch.equal(bufs[0][:, :, :t], before), f"step {t} wrote lookahead keys"
    assert wrote >= 2
    got = torch.cat(outs, 2)
    assert_close(got, ref_out[:, :, t0:], dtype, "decode out", 1e-3)
    H().castle_decode_flush(bufs[0], bufs[1], L, H().make_deferred(*rings, t0), s)
    if dtype == torch.float32:
        assert_close(bufs[0][:, :, :L], ref_U, dtype, "U after the flush", 1e-3)
    else:   # fewer roundings than the step-by-step mode: closer to the fp64 keys
        err_def = (bufs[0][:, :, :L].cpu().double() - ref_U).norm()
        err_plain = (plain[0][:, :, :L].cpu().double() - ref_U).norm()
        assert err_def <= 1.05 * err_plain


@pytest.mark.parametrize("t0,steps,d,rotary", [(0, 21, 64, False), (150, 30, 32, True), (96, 14, 128, False)])
def test_decode_with_half_precision_lookahead_keys(t0, steps, d, rotary):
    """CASTLE_FLAG_U_HALF: a bf16 cache whose lookahead-key buffer holds fp16 bits of U / 64.  The
    forward's U output comes in that format, every step's output equals the oracle's, the flushed
    buffer decodes (64 * fp16) to the oracle's keys, and it does so more closely than the same steps
    on a plain bf16 buffer (11 instead of 8 significant bits per write-back)."""
    from lookahead_keys_attention_amd import _native as N

    B, Hh, dtype = 2, 2, torch.bfloat16
    L = t0 + steps
    ops, _ = rand_ops(B, Hh, L, d, dtype, seed=11 * L + d)
    s = d ** -0.5
    pos = torch.arange(L)
    ref = [t.double() if (idx == 2 or not rotary) else O.rope(t.double(), pos) for idx, t in enumerate(ops)]
    ref_out, ref_U = O.parallel_core(*ref, s, want_U=True)
    dev_ops = [t.to(DEV) for t in ops]

    def fresh(half):
        bufs = [torch.zeros(B, Hh, L + 3, d, dtype=dtype, device=DEV) for _ in range(4)]
        if t0:
            proj = torch.stack([dev_ops[i][:, :, :t0] for i in (3, 4, 5, 0, 1, 2)], 0)   # qu, ku, vu, qc, kc, vc
            proj = proj.permute(1, 3, 0, 2, 4).reshape(B, t0, 6 * Hh * d).contiguous()
            _, U0 = H().castle_attention_packed(proj, Hh, s, True, rotary=rotary, u_half=half)
            bufs[0][:, :, :t0] = U0
            for buf, src in zip(bufs[1:], (ref[3], ref[1], ref[2])):
                buf[:, :, :t0] = src[:, :, :t0].to(dtype).to(DEV)
        return bufs

    half, plain = fresh(True), fresh(False)
    if t0:   # the forward wrote the same keys in the two formats
        U0_ref = O.parallel_core(*[t[:, :, :t0] for t in ref], s, want_U=True)[1]
        assert_close(H().decode_lookahead_keys(half[0][:, :, :t0]), U0_ref, dtype, "prefill U (half format)", 1e-3)
    rings = [[torch.zeros(B, Hh, N.DECODE_DEFER, d, dtype=dtype, device=DEV),
              torch.zeros(B, Hh, L + 3, N.DECODE_DEFER, dtype=torch.float32, device=DEV)] for _ in range(2)]
    ws = H().decode_workspace(B, Hh, d, DEV)
    outs = []
    for t in range(t0, L):
        tok = [x[:, :, t:t + 1] for x in dev_ops]
        o = torch.empty(B, Hh, 1, d, dtype=dtype, device=DEV)
        H().castle_decode_step_hip(*half, t, *tok, s, o, ws, rotary=rotary, deferred=H().make_deferred(*rings[0], t0), u_half=True)
        H().castle_decode_step_hip(*plain, t, *tok, s, torch.empty_like(o), ws, rotary=rotary, deferred=H().make_deferred(*rings[1], t0))
        outs.append(o)
    assert_close(torch.cat(outs, 2), ref_out[:, :, t0:], dtype, "decode out", 1e-3)
    H().castle_decode_flush(half[0], half[1], L, H().make_deferred(*rings[0], t0), s, u_half=True)
    H().castle_decode_flush(plain[0], plain[1], L, H().make_deferred(*rings[1], t0), s)
    got = (half[0][:, :, :L].view(torch.float16).double().cpu() * 64.0)
    err_half = ((got - ref_U).norm() / ref_U.norm()).item()
    err_plain = ((plain[0][:, :, :L].double().cpu() - ref_U).norm() / ref_U.norm()).item()
    assert err_half <= 1.5e-3, f"half-precision keys: {err_half:.3e}"
    assert err_half <= 0.5 * err_plain, f"half format {err_half:.3e} vs bf16 {err_plain:.3e}"
    # the rows the steps appended are zero in both formats, and fp16 / fp32 tensors reject the flag
    with pytest.raises(RuntimeError):
        f16 = [b.half() for b in plain]
        H().castle_decode_step_hip(*f16, L, *[x[:, :, :1].half() for x in dev_ops], s, torch.empty(B, Hh, 1, d, dtype=torch.float16, device=DEV),
                                   ws, u_half=True)



def test_flush_then_step_needs_the_base_moved_to_the_row_count():
    """castle_decode_flush folds the pending sources into U and leaves the castle_deferred struct alone:
    the caller moves `base` to the row count.  Steps that follow a flush with the base moved equal the
    steps of a cache that was never flushed; with the old base the pending terms would be added twice
    (shown here on the stored keys, which is why the header calls the update a postcondition)."""
    from lookahead_keys_attention_amd import _native as N

    B, Hh, d, dtype, t0, t_flush, L = 1, 2, 32, torch.float32, 8, 14, 21
    ops, _ = rand_ops(B, Hh, L, d, dtype, seed=5)
    s = d ** -0.5
    ref = [t.double() for t in ops]
    ref_out, ref_U = O.parallel_core(*ref, s, want_U=True)
    _, U0 = O.parallel_core(*[t[:, :, :t0] for t in ref], s, want_U=True)
    dev_ops = [t.to(DEV) for t in ops]
    ws = H().decode_workspace(B, Hh, d, DEV)

    def run(flush, move_base):
        bufs = [torch.zeros(B, Hh, L + 3, d, dtype=dtype, device=DEV) for _ in range(4)]
        for buf, src in zip(bufs, (U0, ref[3][:, :, :t0], ref[1][:, :, :t0], ref[2][:, :, :t0])):
            buf[:, :, :t0] = src.to(dtype).to(DEV)
        rings = [torch.zeros(B, Hh, N.DECODE_DEFER, d, dtype=dtype, device=DEV),
                 torch.zeros(B, Hh, L + 3, N.DECODE_DEFER, dtype=torch.float32, device=DEV)]
        base, outs = t0, []
        for t in range(t0, L):
            if flush and t == t_flush:
                assert t % N.DECODE_DEFER != 0   # something is pending here
                H().castle_decode_flush(bufs[0], bufs[1], t, H().make_deferred(*rings, base), s)
                if move_base:
                    base = t
            o = torch.empty(B, Hh, 1, d, dtype=dtype, device=DEV)
            H().castle_decode_step_hip(*bufs, t, *[x[:, :, t:t + 1] for x in dev_ops], s, o, ws, deferred=H().make_deferred(*rings, base))
            outs.append(o)
        H().castle_decode_flush(bufs[0], bufs[1], L, H().make_deferred(*rings, base), s)
        return torch.cat(outs, 2), bufs[0][:, :, :L].clone()

    out_plain, U_plain = run(False, False)
    out_moved, U_moved = run(True, True)
    assert_close(out_plain, ref_out[:, :, t0:], dtype, "never flushed", 1e-3)
    assert (out_moved - out_plain).abs().max() <= 1e-5 and (U_moved - U_plain).abs().max() <= 1e-5
    assert_close(U_moved, ref_U, dtype, "U, base moved after the flush", 1e-3)
    _, U_stale = run(True, False)
    assert (U_stale.cpu().double() - ref_U).abs().max() > 1e-2   # the pending terms went in twice


def test_half_precision_lookahead_keys_saturate_instead_of_overflowing():
    """Lookahead keys beyond the window of the half-precision cache format (|U| > 4.2e6) are stored
    saturated, never as infinities: the steps stay finite (each output row a convex combination of
    value rows) and the keys inside the window are still the oracle's.  (Lookahead scores built from
    keys of that size are millions wide; no 16-bit cache resolves them, so the outputs themselves are
    not compared here.)"""
    from lookahead_keys_attention_amd import _native as N

    B, Hh, d, L, dtype = 1, 2, 32, 260, torch.bfloat16
    ops, _ = rand_ops(B, Hh, L, d, dtype, seed=77)
    ops[5] = (ops[5].float().abs() * 6.0e4 + 2.0e4).clamp(0, 6.5e4).to(dtype)     # vu: a few hundred of these add up past 4.2e6
    s = d ** -0.5
    ref_out, ref_U = O.parallel_core(*[t.double() for t in ops], s, want_U=True)
    assert ref_U.abs().max() > 4.5e6
    dev_ops = [t.to(DEV) for t in ops]
    bufs = [torch.zeros(B, Hh, L + 1, d, dtype=dtype, device=DEV) for _ in range(4)]
    rings = [torch.zeros(B, Hh, N.DECODE_DEFER, d, dtype=dtype, device=DEV),
             torch.zeros(B, Hh, L + 1, N.DECODE_DEFER, dtype=torch.float32, device=DEV)]
    ws = H().decode_workspace(B, Hh, d, DEV)
    outs = []
    for t in range(L):
        o = torch.empty(B, Hh, 1, d, dtype=dtype, device=DEV)
        H().castle_decode_step_hip(*bufs, t, *[x[:, :, t:t + 1] for x in dev_ops], s, o, ws,
                                   deferred=H().make_deferred(*rings, 0), u_half=True)
        outs.append(o)
    got = torch.cat(outs, 2)
    assert torch.isfinite(got).all()
    assert got.float().abs().max() <= dev_ops[2].float().abs().max() * 1.01
    H().castle_decode_flush(bufs[0], bufs[1], L, H().make_deferred(*rings, 0), s, u_half=True)
    stored = bufs[0][:, :, :L].view(torch.float16).float().cpu() * 64.0
    assert torch.isfinite(stored).all() and stored.abs().max() <= 65504.0 * 64.0
    small = ref_U.abs() < 4.0e6     # inside the window the keys are the oracle's
    assert ((stored.double() - ref_U)[small].abs() <= 2e-3 * ref_U.abs().max()).all()

