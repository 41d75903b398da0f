"""What the kNN candidate kernel's certificate takes for granted of its operands (no GPU): three
bf16 terms hold an FP32 value exactly, and the three products of them that are left out are at
most 2^-24 of the whole."""
import torch


def _terms(x):
    h = x.to(torch.bfloat16).to(torch.float32)
    m = (x - h).to(torch.bfloat16).to(torch.float32)
    return h, m, (x - h - m).to(torch.bfloat16).to(torch.float32)


def test_three_terms():
    gen = torch.Generator().manual_seed(3)
    n = 1 << 20
    x, q = ((torch.rand(n, generator=gen) + 1) * 2.0 ** torch.randint(-20, 20, (n,), generator=gen)
            * (1 - 2 * torch.randint(0, 2, (n,), generator=gen)) for _ in range(2))
    # all ones in the places that round the furthest, and halves between two bf16 values
    x[:4] = torch.tensor([1 + 127 / 256, 1 + 1 / 256, 2 - 2.0 ** -23, 1 + 2.0 ** -8 + 2.0 ** -17])
    (xh, xm, xl), (qh, qm, ql) = _terms(x), _terms(q)
    assert torch.equal(xh.double() + xm.double() + xl.double(), x.double())
    kept = sum(a.double() * b.double() for a, b in ((xl, qh), (xm, qm), (xh, ql), (xm, qh), (xh, qm), (xh, qh)))
    left = (x.double() * q.double() - kept).abs()
    assert bool((left <= 2.0 ** -24 * (1 + 2.0 ** -9) * (x.double() * q.double()).abs()).all())
    assert torch.equal(torch.stack(_terms(torch.tensor([-0.5]))).flatten(), torch.tensor([-0.5, 0.0, 0.0]))
