"""LM-head confidence (fdl_softmax_confidence) against the float64 torch code it replaces
(generate.py:218, :320, :337): max(softmax(logits.double())) and its index, and the
softmax probability of a given token. The reference is torch's float64 softmax on the CPU:
the float64 terms are identical, or (many values) exp(x) in place of exp(x - m), and the order
of the sum differs, so probabilities agree to ~1e-13 relative and indices exactly. (torch's float64 softmax kernel on this ROCm
build is itself ~1e-9 off the CPU result, so it is not the reference here.)"""
import numpy as np
import pytest
import torch
import torch.nn.functional as F

from fdl import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("rows,vocab,std", [(1, 8, 1.0), (37, 126464, 0.02), (256, 126464, 3.0),
                                            (5, 4096, 30.0)])
def test_softmax_confidence_max_matches_torch_float64(rows, vocab, std):
    gen = torch.Generator().manual_seed(rows + vocab)
    logits = (torch.randn(rows, vocab, generator=gen) * std).to(torch.bfloat16)
    # ties at the maximum: the first index must win
    if vocab > 8:
        logits[0, 5] = logits[0, vocab - 3] = logits[0].max() + 1.0
    ref_p, ref_i = torch.max(F.softmax(logits.to(torch.float64), dim=-1), dim=-1)
    prob, arg = ops.softmax_confidence(logits.to(DEV))
    torch.cuda.synchronize()
    torch.testing.assert_close(prob.cpu(), ref_p, rtol=1e-12, atol=0)
    assert torch.equal(arg.cpu(), ref_i)
    if vocab > 8:
        assert int(arg[0]) == 5


def test_softmax_confidence_token_probability():
    gen = torch.Generator().manual_seed(7)
    rows, vocab = 40, 126464
    logits = (torch.randn(rows, vocab, generator=gen) * 2.0).to(torch.bfloat16)
    tok = torch.randint(0, vocab, (rows,), generator=gen)
    tok[3] = -1  # outside the vocabulary: probability 0
    ref = F.softmax(logits.to(torch.float64), dim=-1).gather(1, tok.clamp(min=0)[:, None]).view(-1)
    ref[3] = 0.0
    prob, _ = ops.softmax_confidence(logits.to(DEV), tok.to(DEV))
    torch.cuda.synchronize()
    torch.testing.assert_close(prob.cpu(), ref, rtol=1e-12, atol=1e-300)


@pytest.mark.parametrize("vocab", [1024, 16384, 126464, 532488])
@pytest.mark.parametrize("token", [False, True])
def test_softmax_confidence_non_finite_rows_match_torch(vocab, token):
    """Rows of all -inf, with a NaN, with a +inf, and with the maximum tied at several
    places: the probability and index are torch.max(softmax(float64)) of the row (NaN and
    index 0 for the rows whose softmax is NaN; the first index of a tie). NaN and +inf stand in a
    row's first and last values (532488: past the chunks that the tabulated kernel can put off),
    and the NaN also in a row whose maximum forces a second pass."""
    x = torch.randn((9, vocab), generator=torch.Generator().manual_seed(3)).to(torch.bfloat16)
    x[0] = float("-inf")
    x[1, 300] = float("nan")
    x[2, 700] = float("inf")
    x[3, vocab - 2] = float("nan")
    x[4, vocab - 2] = float("inf")
    x[5, 300], x[5, 20] = float("nan"), 500.0
    x[6, vocab - 2], x[6, 20] = float("nan"), -float("inf")
    x[7, 10] = x[7, 500] = x[7, 900] = 8.0  # tied maximum
    x[8] = float("-inf")
    x[8, 600] = -3.0                        # one value only
    tok = torch.tensor([5, 300, 700, 9, 9, 20, 3, 500, 600])
    prob, arg = ops.softmax_confidence(x.to(DEV), tok.to(DEV) if token else None)
    p = torch.softmax(x.double(), dim=-1)
    ref_p, ref_i = torch.max(p, dim=-1)
    if token:
        ref_p = p.gather(1, tok[:, None]).view(-1)
    got_p, got_i = prob.cpu(), arg.cpu()
    assert torch.equal(got_i, ref_i), (got_i, ref_i)
    assert torch.isnan(got_p[:7]).all() and torch.isnan(ref_p[:7]).all()
    np.testing.assert_allclose(got_p[7:].numpy(), ref_p[7:].numpy(), rtol=1e-12)
    assert got_p[8] == 1.0


@pytest.mark.parametrize("vocab", [16376, 16384, 16392, 24568, 32776, 131080, 532488])
@pytest.mark.parametrize("token", [False, True])
def test_softmax_confidence_kernel_edges(vocab, token):
    """Vocabulary sizes around the one at which the tabulated kernel takes over, at its chunk
    counts' edges and past the 64 chunks of a thread that it can put off, on rows that hold the
    edges of the tabulated range of magnitudes ([2^-10, 2^6)) and values outside it (zeros,
    denormals, -inf, large ones), and rows whose maximum lies outside it (a second pass). The
    terms are the reference's to an ulp or two of float64 and only the order of up to 532488
    positive terms differs: 1e-12 relative."""
    gen = torch.Generator().manual_seed(vocab)
    x = (torch.randn(7, vocab, generator=gen) * 3.0).to(torch.bfloat16)
    edge = torch.tensor([0.0, -0.0, 2.0**-10, -2.0**-10, 2.0**-10 * (1 - 2.0**-8), 1e-40, -1e-40,
                         63.75, -63.75, -64.0, -700.0, -3e38, float("-inf")]).to(torch.bfloat16)
    x[1, 40:40 + len(edge)] = edge
    x[1, vocab - len(edge):] = edge
    x[2] = (x[2].float() * 40.0).to(torch.bfloat16)  # most values past the table
    x[3] = 0.0                                         # nothing in the table, all tied
    x[4] = (x[4].float() - 400.0).to(torch.bfloat16)  # sums of exp(x) vanish
    x[5, vocab - 1] = 900.0                            # exp(x) overflows
    x[6, 3] = 64.0                                     # the first maximum outside the range
    tok = torch.tensor([vocab - 1, 41, int(x[2].argmax()), vocab, 9, vocab - 1, 3])
    p = F.softmax(x.double(), dim=-1)
    ref_p, ref_i = torch.max(p, dim=-1)
    if token:
        ref_p = p.gather(1, tok.clamp(max=vocab - 1)[:, None]).view(-1)
        ref_p[3] = 0.0
    prob, arg = ops.softmax_confidence(x.to(DEV), tok.to(DEV) if token else None)
    torch.testing.assert_close(prob.cpu(), ref_p, rtol=1e-12, atol=0)
    assert torch.equal(arg.cpu(), ref_i)


@pytest.mark.parametrize("vocab", [1024, 16384])
def test_softmax_confidence_of_a_certain_row_is_exactly_one(vocab):
    """A row whose maximum holds everything (the rest at least 69 below it: less than 2^-53 of the
    sum) has probability 1.0, and one whose maximum is tied 0.5, as float64 softmax gives: for
    every magnitude from 2^-11 to 2^7 in bf16 and both signs (the tabulated maxima and those
    around them), so such rows stay tied with each other and pass a threshold of 1."""
    bits = torch.arange(116 << 7, 134 << 7)
    m = torch.cat((bits, bits | 0x8000)).to(torch.int16).view(torch.bfloat16).to(DEV)
    gen = torch.Generator(device=DEV).manual_seed(vocab)
    for top in m.split(1536):
        rows = len(top)
        low = torch.rand((rows, vocab), generator=gen, device=DEV) * 6.0 + 70.0
        x = (top.float()[:, None] - low).to(torch.bfloat16)
        at = torch.randint(0, vocab, (rows,), generator=gen, device=DEV)
        r = torch.arange(rows, device=DEV)
        x[r, at] = top
        for token in (None, at):
            prob, arg = ops.softmax_confidence(x, token)
            assert (prob == 1.0).all(), (prob.min(), prob.max())
            assert torch.equal(arg, at)
        x[r, (at + 7) % vocab] = top
        assert (ops.softmax_confidence(x)[0] == 0.5).all()
