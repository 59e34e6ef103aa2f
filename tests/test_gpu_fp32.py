"""fp32 tensors: as exact as fp32 sums, element by element, and in the range of fp32."""
import pytest
import torch

pytestmark = pytest.mark.gpu

from oracle import castle_oracle as O

DEV = "cuda:0"


def H():
    from lookahead_keys_attention_amd import ops

    return ops


def operands(B, Hh, L, d, seed, std=0.6):
    g = torch.Generator().manual_seed(seed)
    return [torch.randn(B, Hh, L, d, generator=g) * std for _ in range(6)], torch.randn(B, Hh, L, d, generator=g)


def results(ops, dout, d):
    leaves = [t.to(DEV).requires_grad_() for t in ops]
    out, U = H().castle_attention_hip(*leaves, d ** -0.5, True)
    out.backward(dout.to(DEV))
    return [out.detach(), U] + [t.grad for t in leaves]


def reference(ops, dout, d):
    o64 = [t.double() for t in ops]
    return list(O.parallel_core(*o64, d ** -0.5, want_U=True)) + list(O.closed_form_grads(*o64, d ** -0.5, dout.double()))


def check(got, want, L):
    # fp32 sums of L terms, through three contractions and an exponential: 4 sqrt(L) roundings of 2^-24 (measured: at most half of it)
    for name, a, r in zip(("out", "U", "dqc", "dkc", "dvc", "dqu", "dku", "dvu"), got, want):
        rel = ((a.cpu().double() - r).norm() / r.norm()).item()
        assert rel <= 4 * L ** 0.5 * 2 ** -24, f"{name}: {rel:.2e}"


@pytest.mark.parametrize("B,Hh,L,d", [(1, 2, 127, 64), (1, 2, 128, 64), (2, 2, 129, 32), (1, 3, 159, 16), (1, 2, 161, 64), (1, 1, 192, 64), (2, 1, 225, 32),
                                      (1, 2, 257, 16), (1, 1, 511, 64), (1, 1, 1000, 64), (3, 45, 130, 32)])
def test_results_at_tile_edges(B, Hh, L, d):
    ops, dout = operands(B, Hh, L, d, seed=L + d)
    check(results(ops, dout, d), reference(ops, dout, d), L)


# fewer rows than a tile's worth in so many heads that the scan, and from 513 on the attention, goes by 128 rows a workgroup
@pytest.mark.parametrize("B,Hh,L,d", [(20, 16, 25, 64), (19, 31, 33, 32), (24, 24, 9, 16), (13, 41, 97, 64)])
def test_many_heads_of_few_rows(B, Hh, L, d):
    ops, dout = operands(B, Hh, L, d, seed=L + d)
    check(results(ops, dout, d), reference(ops, dout, d), max(L, 64))   # (below 64 rows the head dimension has the longest sums)


@pytest.mark.parametrize("flag", ["FLAG_RECOMPUTE_SCORES", "FLAG_RECOMPUTE_STATE"])
def test_results_without_tiles_and_without_snapshots(flag, monkeypatch):
    from lookahead_keys_attention_amd import _native

    monkeypatch.setattr(H(), "DEFAULT_FLAGS", getattr(_native, flag))
    ops, dout = operands(2, 2, 300, 64, seed=5)
    check(results(ops, dout, 64), reference(ops, dout, 64), 300)


def test_operands_of_any_magnitude():
    """Heads of very different sizes, and rows of a head."""
    ops, dout = operands(1, 3, 200, 64, seed=6)
    size = torch.tensor([1e-8, 1.0, 1e8])[None, :, None, None]
    ops[2] = ops[2] * size                                   # values
    ops[0], ops[1] = ops[0] / size, ops[1] * size            # the scores stay
    ops[4], ops[3] = ops[4] * size, ops[3] / size            # the gates stay
    ops[5] = ops[5] * size                                   # the lookahead scores stay
    dout = dout * torch.where(torch.arange(200) < 96, 1e-9, 1e3)[None, None, :, None]
    got, want = results(ops, dout, 64), reference(ops, dout, 64)
    for h in range(3):
        check([t[:, h] for t in got], [t[:, h] for t in want], 200)
    rows = slice(0, 96)   # their own gradient of the queries, not only beside that of the large rows
    for h in range(3):
        a, r = got[2][:, h, rows].cpu().double(), want[2][:, h, rows]
        assert (a - r).norm() <= 4 * 200 ** 0.5 * 2 ** -24 * r.norm()


@pytest.mark.parametrize("power", [-80, -30, 60])
def test_gradients_are_linear_in_powers_of_two(power):
    ops, dout = operands(1, 2, 200, 32, seed=7)
    one, other = results(ops, dout, 32), results(ops, dout * 2.0 ** power, 32)
    for a, b in zip(one[2:], other[2:]):
        assert torch.equal(a * 2.0 ** power, b)


def close_by_part(got, want, dim, parts, bound):
    """Each of these rows (dim -2) or columns (-1) by itself, not only beside the larger ones."""
    a, r = got.cpu().double().movedim(dim, 0)[parts], want.movedim(dim, 0)[parts]
    rel = (a - r).flatten(1).norm(dim=1) / r.flatten(1).norm(dim=1)
    assert torch.all(rel <= bound), (rel.max().item(), bound)


# A row of dS is a difference of two sums of about its size: their errors weigh up to a few times as much in it as in the sums, 16 sqrt(L) roundings of 2^-24
SMALL = 16 * 200 ** 0.5 * 2 ** -24


@pytest.mark.parametrize("size", [1e-9, 1e-15])
def test_small_rows_and_columns_beside_large_ones(size):
    """Every second row, or one of 64 columns, is far smaller than its neighbours: an element is held to 2^-24 of itself."""
    L, small = 200, slice(1, None, 2)
    rows = torch.ones(L, 1)
    rows[small] = size
    ops, dout = operands(1, 2, L, 64, seed=8)
    by_row = dout * rows
    got, want = results(ops, by_row, 64), reference(ops, by_row, 64)
    close_by_part(got[2], want[2], -2, small, SMALL)            # dqc of a row follows its dO
    close_by_part(got[4], want[4], -2, [L - 1], SMALL)          # the last key is seen by the last query alone
    columns = torch.ones(64)
    columns[3] = size
    for n in (2, 5):                                            # values, and what the lookahead keys sum
        changed = list(ops)
        changed[n] = ops[n] * columns
        got, want = results(changed, dout, 64), reference(changed, dout, 64)
        close_by_part(got[0 if n == 2 else 1][:, :, :L - 1], want[0 if n == 2 else 1][:, :, :L - 1], -1, [3], SMALL)
        changed[n] = ops[n] * rows.flip(0)                      # row 0 is small, and the last one
        got, want = results(changed, dout, 64), reference(changed, dout, 64)
        if n == 2:
            close_by_part(got[0], want[0], -2, [0], SMALL)
    changed = [ops[0] * rows, *ops[1:]]
    got, want = results(changed, dout, 64), reference(changed, dout, 64)
    close_by_part(got[3], want[3], -2, [L - 1], SMALL)          # dkc of the last key: one row of qc


@pytest.mark.parametrize("score", [-12.0, -40.0])
def test_small_weights_and_gates(score):
    """A key that no query attends to strongly, and gates that are nearly closed, have results of their own."""
    L, d, key = 200, 64, 40
    bound = SMALL + abs(score) * 2 ** -20   # a score is held to a few roundings of 2^-24 of its largest summand, and goes into an exponent
    ops, dout = operands(1, 2, L, d, seed=9)
    weights = [t.clone() for t in ops]
    weights[0][..., 0] = 1.0
    weights[1][:, :, key, 0] = score * d ** 0.5
    got, want = results(weights, dout, d), reference(weights, dout, d)
    close_by_part(got[4], want[4], -2, [key], bound)
    gates = [t.clone() for t in ops]
    gates[3][..., 0] = 1.0
    gates[4][..., 0] = score * d ** 0.5
    got, want = results(gates, dout, d), reference(gates, dout, d)
    for n in (1, 5, 7):   # U, dqu, dvu
        close_by_part(got[n][None], want[n][None], 0, [0], bound)


@pytest.mark.parametrize("L", [100, 200])
@pytest.mark.parametrize("sign", [-1.0, 1.0])
def test_infinite_elements_of_the_forward_pass(L, sign):
    """An infinite source element opens or closes its gates, a key whose score is -inf has no weight: results stay finite."""
    ops, _ = operands(1, 2, L, 64, seed=10)
    ops[3][..., 0], ops[0][..., 0] = 0.5, 0.5
    infinite, far = [t.clone() for t in ops], [t.clone() for t in ops]
    for to, x in ((infinite, float("inf")), (far, 1e30)):
        to[4][:, :, 70, 0] = sign * x
        to[1][:, :, 5, 0] = -x
    with torch.no_grad():
        out, U = H().castle_attention_hip(*[t.to(DEV) for t in infinite], 0.125, True)
    want, want_U = O.parallel_core(*[t.double() for t in far], 0.125, want_U=True)
    check((out, U), (want, want_U), L)
