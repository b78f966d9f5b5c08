"""float16 attention in tiles of 256 query rows: probabilities against one reference per row, the largest score of the
first 64 keys, and the online softmax where a later score is beyond what that leaves."""

import pytest
import torch

pytestmark = pytest.mark.gpu

# Queries and probabilities are rounded to 2^-11 of themselves at most, the output too: random errors of about a third of
# that each (4.1e-4 measured for all together); scores of up to 40 carry the queries' rounding into the exponent where the
# online softmax takes over, 40 * 2^-11 / 3.
TOL = 8e-3


def _reference(q, k, v, extra=None):
    s = q.double() @ k.double().transpose(-1, -2) / q.shape[-1] ** 0.5
    if extra is not None:
        s = s + extra
    return s.softmax(-1) @ v.double(), torch.logsumexp(s, -1)


def _rel(a, b):
    return float((a.double() - b).norm() / b.norm())


# keys: one, short of, at and past the first tile of 64, several tiles; the step in the scores (natural) behind the first 64
# keys: none, inside, at the edge of and beyond 16 powers of two, and far below
@pytest.mark.parametrize("Nc", [1, 63, 64, 65, 200, 1100])
@pytest.mark.parametrize("step", [0.0, 9.0, 11.1, 12.0, 14.0, 40.0, -40.0])
def test_context_with_a_step_in_its_scores(device, tuning, Nc, step):
    import ar_nanotabpfn_amd.attention_kernels as ak

    tuning(ARTAB_SMALL=0)
    B, H, Dh = 300, 2, 32
    g = torch.Generator().manual_seed(Nc)
    q = torch.randn(B, H, 1, Dh, generator=g)
    k, v = (torch.randn(H, Nc, Dh, generator=g) for _ in range(2))
    q[..., 0] = 4.0  # the first element makes the step, the same for every query
    k[..., 0] = 0.0
    k[:, 64:, 0] = step * Dh ** 0.5 / 4.0
    q, k, v = (t.to(device, torch.float16) for t in (q, k, v))
    out, lse = ak.context_attention(q, k, v)
    want, want_lse = _reference(q, k, v)
    assert _rel(out, want) <= TOL
    assert float((lse.double() - want_lse).abs().max()) <= 2 * TOL * max(1.0, abs(step))


# one key among the first 64 that is `up` (natural) above a long tail, all of one score or with a spread of them: 2^-11 to
# 2^-20 of its probability each, which 16 bits hold in steps of 2^-24
@pytest.mark.parametrize("up", [8.0, 10.0, 11.0, 12.0, 14.0])
@pytest.mark.parametrize("spread", [0.0, 1.0])
def test_one_early_key_above_a_long_tail(device, tuning, up, spread):
    import ar_nanotabpfn_amd.attention_kernels as ak

    tuning(ARTAB_SMALL=0, ARTAB_SPLIT=1)
    B, H, Nc, Dh = 300, 1, 16384, 32
    g = torch.Generator().manual_seed(int(up))
    q = spread * torch.randn(B, H, 1, Dh, generator=g)
    k, v = (torch.randn(H, Nc, Dh, generator=g) for _ in range(2))
    q[..., 0] = 4.0
    k[..., 0] = 0.0
    k[:, 17, 0] = up * Dh ** 0.5 / 4.0
    q, k, v = (t.to(device, torch.float16) for t in (q, k, v))
    errors = []
    want, want_lse = _reference(q, k, v)
    for lean in (1, 0):  # 0: the online softmax
        tuning(ARTAB_LEAN=lean)
        out, lse = ak.context_attention(q, k, v)
        errors.append((_rel(out, want), float((lse.double() - want_lse).abs().max())))
    # the same probabilities in the same steps; beside them the output's rounding, 2^-11, a third of it on average, and the
    # logarithm's in float32, 2^-24 of a sum in front of which up to `up` is subtracted
    assert errors[0][0] <= 1.1 * errors[1][0] + 2.0 ** -11 / 3
    assert errors[0][1] <= 1.1 * errors[1][1] + 4 * up * 2.0 ** -24


def test_rows_of_no_use_for_a_reference(device, tuning):
    """Scores of minus infinity in the first tile, all of them, or one that is not a number: as the online softmax has them."""
    import ar_nanotabpfn_amd.attention_kernels as ak

    tuning(ARTAB_SMALL=0)
    B, H, Nc, Dh = 260, 1, 130, 32
    q = torch.randn(B, H, 1, Dh, device=device).half()
    k, v = (torch.randn(H, Nc, Dh, device=device).half() for _ in range(2))
    q[..., 0] = 1.0
    k[:, :64, 0] = -float("inf")
    out, lse = ak.context_attention(q, k, v)
    want, want_lse = _reference(q, k[:, 64:], v[:, 64:])
    assert _rel(out, want) <= TOL and float((lse.double() - want_lse).abs().max()) <= 2 * TOL
    k[:, 64:, 0] = -float("inf")
    out, lse = ak.context_attention(q, k, v)
    assert torch.equal(out, torch.zeros_like(out)) and torch.isneginf(lse).all()
    k[:, :, 0] = 0
    q[7, 0, 0, 3] = float("nan")
    out, _ = ak.context_attention(q, k, v)
    others = torch.arange(B, device=device) != 7
    want, _ = _reference(q[others], k, v)
    assert _rel(out[others], want) <= TOL and torch.isnan(out[7]).all()


@pytest.mark.parametrize("Nc,Nt", [(1, 130), (40, 150), (64, 129), (500, 140)])
def test_teacher_forcing_in_wide_tiles(device, tuning, Nc, Nt):
    import ar_nanotabpfn_amd.attention_kernels as ak
    from oracle import attention_oracle as ao

    tuning(ARTAB_BM=256)
    B, H, Dh = 2, 2, 32
    q, kc, vc, kb, vb = (torch.randn(*s, device=device).half() for s in
                         ((B, H, 2 * Nt, Dh), (B, H, Nc, Dh), (B, H, Nc, Dh), (B, H, Nt, Dh), (B, H, Nt, Dh)))
    out = ak.teacher_forcing_attention(q, kc, vc, kb, vb, Nt)
    want = torch.from_numpy(ao.hybrid_teacher_forcing_attention(*(t.double().cpu().numpy() for t in (q, kc, vc, kb, vb)), Nt))
    assert _rel(out.cpu(), want) <= TOL
