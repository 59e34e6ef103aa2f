"""fp32 products on the 16-bit matrix instructions, an element in three bf16 parts (csrc/castle_gemm32.hip)."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def product(*args):
    from lookahead_keys_attention_amd import _native

    return _native.host().product(*args)


def layouts(a, b):
    at, bt = a.t().contiguous(), b.t().contiguous()
    return [(a, False, b, False), (a, False, bt, True), (at, True, bt, True)]


# tiles of 32 and 64 by one to eight waves: remainders in every direction, contractions of less than a step, waves without a step, ranges of the contraction
@pytest.mark.parametrize("M,N,K", [(8, 8, 8), (24, 40, 24), (64, 64, 32), (72, 136, 40), (256, 512, 512), (96, 3072, 512), (1000, 520, 264), (2504, 2048, 64), (6000, 1032, 104),
                                   (4104, 1024, 264), (72, 64, 5000), (256, 512, 3080)])
def test_no_further_from_64_bits_than_fp32(M, N, K):
    g = torch.Generator(device=DEV).manual_seed(M + K)
    a, b = (torch.randn(*s, generator=g, device=DEV) for s in ((M, K), (N, K)))
    ref, size = a.double() @ b.double().t(), a.double().abs() @ b.double().abs().t()
    for operands in layouts(a, b):
        got = product(*operands, 0, None).double()
        # the parts leave 2^-23 of a product; K sums of 2^-24 each at most, as in fp32
        assert torch.all((got - ref).abs() <= (K + 4) * 2.0 ** -24 * size)
        # and on average: 2^-24 for the result, and a sum that is rounded after every second product, as the fp32 instruction does, adds errors of 2^-24 sqrt(k / 3) of
        # a product's size after k of them: sqrt(K / 12) in all
        assert (got - ref).norm() <= 2.0 ** -24 * (1 + (K / 12) ** 0.5) * ref.norm()
    if N % 64 == 0:
        u = torch.randn(M, N, generator=g, device=DEV)
        act = torch.empty_like(u)
        up = product(a, False, b, False, 1, act).double()
        assert torch.all((up - ref).abs() <= (K + 4) * 2.0 ** -24 * size)
        assert (act.double() - torch.nn.functional.gelu(up)).norm() <= 1e-6 * act.double().norm()


@pytest.mark.parametrize("M,N,K", [(72, 136, 40), (256, 512, 512), (2504, 2048, 64), (4104, 1024, 264), (72, 64, 5000)])
def test_infinities_nans_and_the_ends_of_the_range(M, N, K):
    g = torch.Generator(device=DEV).manual_seed(M)
    a, b = (torch.randn(*s, generator=g, device=DEV) for s in ((M, K), (N, K)))
    a[3, 5], a[M - 1, K - 1], b[N - 2, 7] = float("inf"), float("nan"), float("-inf")
    a[9], b[11] = 0.0, 0.0
    a[9, K // 2] = 3.4028e38   # rounds to infinity in bf16
    a[20, 1], b[30, 1] = 2.0 ** 127, 4.0   # and a sum that leaves the range
    a[40] *= 2.0 ** -100
    want = a.double() @ b.double().t()
    finite = want.abs() <= torch.finfo(torch.float32).max
    for operands in layouts(a, b):
        got = product(*operands, 0, None)
        assert torch.equal(got.isnan(), want.isnan())
        over = ~finite & ~want.isnan()
        assert torch.all(got[over] == torch.sign(want[over]).float() * float("inf"))
        size = a.double().abs() @ b.double().abs().t()
        assert torch.all(((got.double() - want).abs() <= (K + 4) * 2.0 ** -24 * size)[finite])


@pytest.mark.parametrize("M,N,K", [(72, 136, 40), (256, 512, 512), (4104, 1024, 264)])
@pytest.mark.parametrize("power", [-105, -112, -118])
def test_elements_near_the_smallest_normal_number(M, N, K, power):
    """Rows of either operand whose third part, 2^-16 of an element, would be below what bf16 holds."""
    g = torch.Generator(device=DEV).manual_seed(N)
    a, b = (torch.randn(*s, generator=g, device=DEV) for s in ((M, K), (N, K)))
    a[5:40] *= 2.0 ** power
    want, size = a.double() @ b.double().t(), a.double().abs() @ b.double().abs().t()
    for operands in layouts(a, b) + [(b, False, a, False)]:
        got, ref, s = product(*operands, 0, None).double(), want, size
        if operands[0] is b:
            ref, s = want.t(), size.t()
        assert torch.all((got - ref).abs() <= (K + 4) * 2.0 ** -24 * s + K * 2.0 ** -149)
