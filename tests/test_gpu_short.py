"""Forward pass of short sequences without a backward pass: one launch, a workgroup per 32 queries of a head (csrc/castle_short.hip)."""
import pytest
import torch

pytestmark = pytest.mark.gpu

from oracle import castle_oracle as O

DEV = "cuda:0"


def H():
    from lookahead_keys_attention_amd import ops

    return ops


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,Hh,L,d,rotary", [(1, 2, 1, 64, False), (1, 3, 31, 64, True), (2, 2, 32, 32, False), (1, 2, 33, 16, False), (1, 2, 64, 128, False),
                                             (2, 1, 65, 64, True), (1, 2, 96, 128, True), (1, 2, 97, 128, False), (1, 4, 127, 64, False), (5, 7, 128, 64, False),
                                             (2, 2, 128, 32, True), (1, 2, 129, 64, False), (3, 64, 128, 16, False), (3, 65, 128, 16, False), (1, 300, 34, 16, False)])
def test_forward_without_a_graph(B, Hh, L, d, rotary, dtype):
    g = torch.Generator().manual_seed(L + d)
    ops = [(torch.randn(B, Hh, L, d, generator=g) * 0.6).to(dtype) for _ in range(6)]
    with torch.no_grad():
        out, U = H().castle_attention_hip(*[t.to(DEV) for t in ops], d ** -0.5, True, rotary=rotary)
    dev = [t.to(DEV) for t in ops]
    general, general_U = H().castle_attention_hip(*dev, d ** -0.5, True, rotary=rotary)   # with a graph: the general path
    o64 = [t.double() for t in ops]
    if rotary:
        at = torch.arange(L)
        o64 = [t if n == 2 else O.rope(t, at) for n, t in enumerate(o64)]
    ref, ref_U = O.parallel_core(*o64, d ** -0.5, want_U=True)
    for got, other, want in ((out, general, ref), (U, general_U, ref_U)):
        if want.abs().max() == 0:
            assert torch.all(got == 0)
            continue
        err, allowed = [((t.cpu().double() - want).norm() / want.norm()).item() for t in (got, other)]
        # the same roundings of operands and results as the general path: no further from 64 bits than it, up to chance
        assert err <= 1.2 * allowed + 2.0 ** -(9 if dtype == torch.bfloat16 else 12), (err, allowed)


# up to two tiles of 32 rows at any number of heads; beyond, up to 768 workgroups; the rows of four tiles do not fit into LDS at d = 128
@pytest.mark.parametrize("B,Hh,L,d,one", [(1, 2, 1, 64, True), (1, 2, 33, 16, True), (2, 1, 65, 64, True), (1, 2, 96, 128, True), (1, 2, 97, 128, False), (5, 7, 128, 64, True),
                                          (1, 2, 129, 64, False), (3, 64, 128, 16, True), (193, 1, 128, 16, False), (1, 256, 96, 32, True), (1, 257, 96, 32, False), (1, 800, 64, 16, True)])
def test_which_calls_take_one_launch(B, Hh, L, d, one):
    from lookahead_keys_attention_amd import _native as N

    ops = [torch.zeros(B, Hh, L, d, device=DEV, dtype=torch.bfloat16) for _ in range(6)]
    for records, want in ((False, ["attn"] if one else ["prep", "scan", "attn"]), (True, ["prep", "scan", "attn"])):
        N.profile_enable(True)
        try:
            with torch.set_grad_enabled(records):
                H().castle_attention_hip(*ops, d ** -0.5)
            kernels = [name for name, _ in N.profile_read()]
        finally:
            N.profile_enable(False)
        assert kernels == want, (records, kernels)


@pytest.mark.parametrize("half", [False, True])
def test_strided_operands_and_cache_rows(half):
    """The packed projection, and lookahead keys as the first rows of a cache buffer in either format."""
    heads, d, L = 4, 64, 100
    proj = (torch.randn(2, L, 6 * heads * d, generator=torch.Generator().manual_seed(3)) * 0.6).bfloat16().to(DEV)
    with torch.no_grad():
        a, Ua = H().castle_attention_packed(proj, heads, d ** -0.5, True, 160, u_half=half)
    b, Ub = H().castle_attention_packed(proj, heads, d ** -0.5, True, 160, u_half=half)
    if half:
        Ua, Ub = H().decode_lookahead_keys(Ua), H().decode_lookahead_keys(Ub)
    for x, y in ((a, b), (Ua, Ub)):
        assert (x.float() - y.float()).norm() <= 2 ** -8 * y.float().norm()


def test_range_control_and_status():
    """Values whose sums leave the fp16 range, and inputs beyond it: like the general path."""
    ops = [(torch.randn(1, 2, 100, 64, generator=torch.Generator().manual_seed(4)) * 0.6).bfloat16() for _ in range(6)]
    ops[5] = ops[5] * 4e4
    ops[0] = ops[0] * 1e-5
    dev = [t.to(DEV) for t in ops]
    with torch.no_grad():
        a, Ua = H().castle_attention_hip(*dev, 0.125, True)
    ref, ref_U = O.parallel_core(*[t.double() for t in ops], 0.125, want_U=True)
    for x, y in ((a, ref), (Ua, ref_U)):
        assert torch.isfinite(x).all() and (x.cpu().double() - y).norm() <= 2e-2 * y.norm()
    from lookahead_keys_attention_amd import _native as N

    big = [t.clone() for t in dev]
    big[1][0, 1, 5, 3] = 1e5
    for tensors, status in ((dev, 0), (big, 1)):
        ws = torch.ops.castle_hip.attention(*tensors, 0.125, False, N.FLAG_FORWARD_ONLY, False)[2]
        assert H().range_status(ws) == status
