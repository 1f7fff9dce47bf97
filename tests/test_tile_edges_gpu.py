"""The sizes at which the tile kernels' dispatch rules change or a tile, group or split is incomplete, against the oracle.

Bounds: d_hidden and d_weight are bf16-rounded products of a dz that is itself rounded to bf16 once, 2^-9 / sqrt(3) relative
each and independent of the sizes: 3e-3 in the 2-norm, a single row at most four times that where its norm is of the order of the
others'."""

from __future__ import annotations

import pytest
import torch

from oracle import lmhead_oracle as O
from skyrl_amd import _lib, ops
from skyrl_amd import torch_utils as TU
from skyrl_amd.model_utils import from_parallel_hidden_to_logprobs
from skyrl_amd.mtp_soft_ce import (draft_soft_ce_from_hidden, draft_soft_ce_topk_from_hidden, soft_ce_from_hidden, soft_ce_topk_from_hidden,
                                   softce_bwd, softce_fwd, topk_logits_from_hidden)

pytestmark = pytest.mark.gpu

GRAD_REL_L2 = 5e-3
GRAD_ROW_REL_L2 = 2e-2
ERR_WORKSPACE = -4   # include/skyrl_lmhead.h


def _operands(T, H, V, seed, dtype=torch.bfloat16):
    gen = torch.Generator().manual_seed(seed)
    hidden = torch.randn(T, H, generator=gen).to(torch.bfloat16)
    weight = (torch.randn(V, H, generator=gen) * 3 / H**0.5).to(dtype)
    labels = torch.randint(0, V, (T,), generator=gen)
    g, q = torch.randn(T, generator=gen), torch.randn(T, generator=gen) * 0.2
    return hidden, weight, labels, g, q


def _close(got, want, tag):
    got, want = got.detach().double().cpu(), want.double()
    rel = float((got - want).norm() / want.norm())
    norms = want.norm(dim=1)
    row = float(((got - want).norm(dim=1) / norms.clamp_min(0.1 * float(norms.mean()))).max())
    assert rel < GRAD_REL_L2 and row < GRAD_ROW_REL_L2, f"{tag}: {rel:.2e}, worst row {row:.2e}"


# The last group of 128 vocabulary rows is moved back from V = 1024 on: one row left over, one missing, the group in the lower
# and in the upper half of a tile, alone in its chunk, and the sizes around the rule's line.
@pytest.mark.parametrize("V,vc", [(1023, 0), (1025, 0), (1025, 256), (1151, 256), (1152, 256), (1153, 256), (1279, 512), (5001, 0)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_vocabulary_that_ends_inside_a_group(V, vc, dtype, cuda_device):
    T, H, t = 300, 192, 0.8
    hidden, weight, labels, g, q = _operands(T, H, V, seed=V + vc, dtype=dtype)
    labels[:6] = torch.tensor([V - 1, V - 128, V // 128 * 128 - 1, min(V - 1, V // 128 * 128), V - 127, 0])
    g[7::5], q[7::5] = 0.0, 0.0
    h, w, y, gd, qd = (x.to(cuda_device) for x in (hidden, weight, labels, g, q))
    _, _, lse, pz = ops.lmhead_fwd(h, w, y, 1.0 / t, True)
    ex = O.exact_fwd_bwd(hidden, weight, labels, t, g, q)
    for active in (False, True):
        dh, dw = ops.lmhead_bwd(h, w, y, lse, pz, gd, qd, 1.0 / t, vc, active)
        _close(dh, ex["d_hidden"], f"dHidden V={V} chunk={vc}")
        _close(dw, ex["d_weight"], f"dW V={V} chunk={vc}")
    assert torch.equal(ops.lmhead_bwd_hidden(h, w, y, lse, pz, gd, qd, 1.0 / t, vc, True), dh)
    if dtype == torch.bfloat16:
        acc = torch.full((V, H), 0.5, device=cuda_device)
        ops.lmhead_bwd_accumulate(h, w, y, lse, pz, gd, qd, 1.0 / t, acc, vc)
        _close(acc - 0.5, ex["d_weight"], f"accumulated dW V={V}")
        # the draft loss contracts over the same vocabulary
        s = hidden.reshape(2, 150, H).to(cuda_device).requires_grad_(True)
        teacher = torch.randn(2, 150, H, generator=torch.Generator().manual_seed(V)).to(torch.bfloat16)
        up = g.reshape(2, 150)
        (soft_ce_from_hidden(s, teacher.to(cuda_device), w, shift=1, vocab_chunk=vc) * up.to(cuda_device)).sum().backward()
        zs, zt = hidden.double() @ weight.double().t(), teacher.roll(-1, dims=1).reshape(T, H).double() @ weight.double().t()
        want = (g.double()[:, None] * (zs.softmax(-1) - zt.softmax(-1))) @ weight.double()
        _close(s.grad.reshape(T, H), want, f"draft loss V={V}")


# The dHidden contraction is split over workgroups when there are few tiles: one token tile and as many splits as the vocabulary
# allows, several chunks, a last chunk with fewer k-tile pairs than splits (one split has nothing to add), hidden columns that
# overhang a tile, and a count of active rows far below the number of tokens (down to none).
@pytest.mark.parametrize("T,H,V,vc", [(40, 64, 20000, 0), (700, 128, 4224, 2048), (257, 320, 8192, 0), (513, 192, 6001, 2048)])
@pytest.mark.parametrize("keep", [1.0, 0.3, 0.0])
def test_split_hidden_gradient(T, H, V, vc, keep, cuda_device):
    hidden, weight, labels, g, q = _operands(T, H, V, seed=T + V)
    keep_rows = torch.rand(T, generator=torch.Generator().manual_seed(T)) < keep
    g, q = g * keep_rows, q * keep_rows
    h, w, y, gd, qd = (x.to(cuda_device) for x in (hidden, weight, labels, g, q))
    _, _, lse, pz = ops.lmhead_fwd(h, w, y, 1.0, True)
    dense = ops.lmhead_bwd_bf16(h, w, y, lse, pz, gd, qd, 1.0, vc)
    active = ops.lmhead_bwd_bf16(h, w, y, lse, pz, gd, qd, 1.0, vc, True)
    frozen = ops.lmhead_bwd_hidden(h, w, y, lse, pz, gd, qd, 1.0, vc, True)
    if keep == 0.0:
        assert all(not t.any() for t in (*dense, *active, frozen))
        return
    ex = O.exact_fwd_bwd(hidden, weight, labels, 1.0, g, q)
    for dh in (dense[0], active[0], frozen):
        _close(dh, ex["d_hidden"], f"dHidden T={T} H={H} V={V} chunk={vc}")
        assert not dh[(~keep_rows).to(cuda_device)].any()
    for dw in (dense[1], active[1]):
        _close(dw, ex["d_weight"], f"dW T={T} H={H} V={V} chunk={vc}")
    assert torch.equal(active[0], ops.lmhead_bwd_bf16(h, w, y, lse, pz, gd, qd, 1.0, vc, True)[0])   # a fixed order of addition


# Candidates of a later chunk that all beat the first chunk's 31 best: inserted one by one, or merged from 35 keys on in registers of one, four and
# eight keys a lane, and from LDS behind 512; exact sums of two terms, so any order of the keys but torch's would show.
@pytest.mark.parametrize("n", [1, 3, 4, 33, 34, 225, 226, 481, 482, 700])
def test_topk_candidates_that_all_pass(n, cuda_device):
    first, H, k, T = 32768, 64, 31, 3  # the first chunk of so few tokens
    gen = torch.Generator().manual_seed(n)
    weight = torch.zeros(first + n, H)
    weight[:first, 0] = torch.randint(-64, 64, (first,), generator=gen).float()
    late = torch.randperm(n, generator=gen).float()
    weight[first:, 0], weight[first:, 1] = 64 + late // 8, (late % 8) / 8
    hidden = torch.zeros(T, H)
    hidden[:, :2] = 1.0
    values, columns = topk_logits_from_hidden(hidden.to(torch.bfloat16).to(cuda_device), weight.to(torch.bfloat16).to(cuda_device), k)
    logits = weight[:, 0] + weight[:, 1]
    order = sorted(range(first + n), key=lambda v: (-float(logits[v]), v))[:k]  # higher first, lower column first among equals
    assert values.cpu().tolist() == [[float(logits[v]) for v in order]] * T and columns.cpu().tolist() == [order] * T


# Alone in its launch, dHidden goes in equal shares of its tiles where whole workgroups per tile leave CUs idle: a round of 256 tiles and a
# part of one, with tiles of one workgroup among them, three tiles for eight workgroups, both in one chunk and in several of which the last is
# narrow and ends in a moved group, and token counts that the host does not know.  Beside dW the same sums run whole or in splits: fp32 sums of
# V <= 2^15 products in another order, rounded to bf16 once: an element in some 200 falls to the other side, sqrt(1 / 200) 2^-8 = 3e-4.
SHARES = [(4500, 4160, 8000, 0), (4500, 4160, 12300, 8192), (1500, 4096, 32000, 0), (1400, 4096, 32001, 20480)]
NO_ROOM_FOR_SHARES = (4500, 4160, 9300, 4096)  # but for the draft loss


@pytest.mark.parametrize("T,H,V,vc", [*SHARES, NO_ROOM_FOR_SHARES])
@pytest.mark.parametrize("keep", [1.0, 0.7])
def test_hidden_gradient_in_shares(T, H, V, vc, keep, cuda_device):
    hidden, weight, labels, g, q = _operands(T, H, V, seed=T + V)
    keep_rows = torch.rand(T, generator=torch.Generator().manual_seed(T)) < keep
    h, w, y, gd, qd = (x.to(cuda_device) for x in (hidden, weight, labels, g * keep_rows, q * keep_rows))
    _, _, lse, pz = ops.lmhead_fwd(h, w, y, 1.0, True)
    want = ops.lmhead_bwd_bf16(h, w, y, lse, pz, gd, qd, 1.0, vc)[0].float()
    for active in (False, True):
        dh = ops.lmhead_bwd_hidden(h, w, y, lse, pz, gd, qd, 1.0, vc, active)
        assert float((dh.float() - want).norm() / want.norm()) < 1e-3
        assert float((dh.float() - want).abs().max() / want.abs().max()) < 2**-7  # no tile is missing, none added twice
        assert not dh[(~keep_rows).to(cuda_device)].any()
        assert torch.equal(dh, ops.lmhead_bwd_hidden(h, w, y, lse, pz, gd, qd, 1.0, vc, active))  # a fixed order of addition
    s, teacher = h.clone().requires_grad_(True), h.roll(1, 0)
    per_token = soft_ce_from_hidden(s.reshape(1, T, H), teacher.reshape(1, T, H), w)
    per_token.backward(gd.reshape(1, T))
    probs = [torch.softmax(x.float() @ w.t().float(), dim=-1) for x in (h, teacher)]
    dz = (gd.unsqueeze(1) * (probs[0] - probs[1])).to(torch.bfloat16).float()
    ref = dz @ w.float()  # dz rounded to bf16 from probabilities that differ in fp32 roundings, dHidden rounded to bf16: 2^-8 / sqrt(3) each
    assert float((s.grad.float() - ref).norm() / ref.norm()) < 5e-3


# Several blocks of tokens whose contractions the device cuts by one rule, the last with few tiles: 8 and 4 of them in groups of four, cut for 64
# workgroups each.  Tokens without a gradient are moved out of the way, so the last block holds the same number with them.  Against the blocks by
# themselves: the bounds of test_hidden_gradient_in_shares.
SHARES_OF_A_SHORT_LAST_BLOCK = [(33024, 2048, 16000, 0), (33792, 256, 32000, 0)]


@pytest.mark.parametrize("T,H,V,vc", SHARES_OF_A_SHORT_LAST_BLOCK)
@pytest.mark.parametrize("masked", [0, 300])
def test_hidden_gradient_of_a_short_last_block(T, H, V, vc, masked, cuda_device):
    T += masked
    hidden, weight, labels, g, q = _operands(T, H, V, seed=T)
    rest = torch.randperm(T, generator=torch.Generator().manual_seed(T))[:masked]
    g[rest], q[rest] = 0.0, 0.0
    h, w, y, gd, qd = (x.to(cuda_device) for x in (hidden, weight, labels, g, q))
    _, _, lse, pz = ops.lmhead_fwd(h, w, y, 1.0, True)
    dh = ops.lmhead_bwd_hidden(h, w, y, lse, pz, gd, qd, 1.0, vc, True)
    assert not dh[rest.to(cuda_device)].any()
    for first in range(0, T, 4096):
        b = slice(first, first + 4096)
        want = ops.lmhead_bwd_hidden(h[b], w, y[b], lse[b], pz[b], gd[b], qd[b], 1.0, vc, False).float()
        assert float((dh[b].float() - want).norm() / want.norm()) < 1e-3, first
        assert float((dh[b].float() - want).abs().max() / want.abs().max()) < 2**-7, first


# The first vocabulary chunk of the top-k search is stored and searched: its width follows the number of tokens, the later ones the
# room for candidate lists and k.  One chunk only, one column behind the first, many equal logits at the k-th rank, k = V.
@pytest.mark.parametrize("T,H,V,k", [(3, 64, 8192, 5), (300, 64, 32769, 32), (260, 64, 33025, 1000), (2050, 64, 8449, 64), (5, 64, 40, 40)])
@pytest.mark.parametrize("ties", [False, True])
def test_topk_first_chunk(T, H, V, k, ties, cuda_device):
    gen = torch.Generator().manual_seed(T + V)
    hidden = torch.randn(T, H, generator=gen).to(torch.bfloat16)
    weight = torch.randn(V, H, generator=gen).to(torch.bfloat16)
    if ties:  # small whole numbers: exact in bf16 and fp32, each value many times in a row
        hidden = torch.zeros(T, H, dtype=torch.bfloat16)
        hidden[:, 0] = 1.0
        weight[:, 0] = torch.randint(-3, 4, (V,), generator=gen).to(torch.bfloat16)
        weight[V // 2, 0] = float("nan")
    z = hidden.double() @ weight.double().t()
    if ties:
        z = weight[:, 0].double().expand(T, V).clone()
        z[:, V // 2] = -torch.inf
    values, columns = topk_logits_from_hidden(hidden.to(cuda_device), weight.to(cuda_device), k)
    values, columns = values.cpu().double(), columns.cpu()
    if ties:  # value first, then the lower column; the NaN is never taken while numbers are left
        order = torch.argsort(-z[0] * (V + 1) + torch.arange(V), stable=True)[:k]
        n = min(k, V - 1)
        assert torch.equal(columns[:, :n], order[:n].expand(T, n)) and torch.equal(values[:, :n], z[:, order[:n]])
        return
    want = z.topk(min(k, V), dim=1)
    assert float((values - want.values).abs().max()) < 1e-4
    assert float((values - z.gather(1, columns)).abs().max()) < 1e-4
    assert all(len(set(r)) == k for r in columns.tolist())


# The draft loss's backward runs on the tokens with an upstream gradient only: none, one, one 128-token tile, just over one, all.
@pytest.mark.parametrize("active", [0, 1, 128, 129, 600])
@pytest.mark.parametrize("V,vc", [(2304, 0), (5001, 1024)])
def test_draft_loss_backward_on_active_tokens(active, V, vc, cuda_device):
    B, S, H = 3, 200, 128
    hidden, weight, _, g, _ = _operands(B * S, H, V, seed=V + active)
    teacher = torch.randn(B, S, H, generator=torch.Generator().manual_seed(V)).to(torch.bfloat16)
    keep = torch.zeros(B * S)
    keep[torch.randperm(B * S, generator=torch.Generator().manual_seed(active))[:active]] = 1.0
    g = (g * keep).reshape(B, S)
    s = hidden.reshape(B, S, H).to(cuda_device).requires_grad_(True)
    loss = soft_ce_from_hidden(s, teacher.to(cuda_device), weight.to(cuda_device), shift=2, vocab_chunk=vc)
    (loss * g.to(cuda_device)).sum().backward()
    grad = s.grad.reshape(B * S, H)
    assert not grad[(keep == 0).to(cuda_device)].any()
    if active:
        zs = hidden.double() @ weight.double().t()
        zt = teacher.roll(-2, dims=1).reshape(B * S, H).double() @ weight.double().t()
        want = (g.reshape(-1).double()[:, None] * (zs.softmax(-1) - zt.softmax(-1))) @ weight.double()
        _close(grad, want, f"{active} active tokens, V={V}")


# Logits rows that start anywhere: every offset of a row from a 16-byte boundary, rows shorter than the way to it, odd pitches, a
# gradient buffer whose rows start elsewhere than the logits' (single accesses) and one written in place.
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("V,pitch", [(1, 1), (5, 7), (7, 9), (63, 65), (4099, 4099), (9001, 9008)])
def test_logits_rows_at_any_offset(dtype, V, pitch, cuda_device):
    T, t = 9, 0.7
    gen = torch.Generator().manual_seed(V)
    for offset in range(8):
        buf = torch.randn(offset + T * pitch, generator=gen).mul(3).to(dtype).to(cuda_device)
        z = buf[offset:].as_strided((T, V), (pitch, 1))
        labels = torch.randint(0, V, (T,), generator=gen)
        g, q = torch.randn(T, generator=gen), torch.randn(T, generator=gen) * 0.1
        zd = z.detach().cpu().double().requires_grad_(True)
        ls = torch.log_softmax(zd / t, dim=1)
        want_lp, want_ent = ls.gather(1, labels[:, None])[:, 0], -(ls.exp() * ls).sum(1)
        (want_lp * g + want_ent * q).sum().backward()
        lp, ent, lse, pz = TU.logits_fwd(z, labels.to(cuda_device), 1.0 / t, True)
        assert float((lp.cpu().double() - want_lp.detach()).abs().max()) < 1e-5 * (1 + float(want_lp.detach().abs().max()))
        assert float((ent.cpu().double() - want_ent.detach()).abs().max()) < 1e-5 * (1 + float(want_ent.detach().abs().max()))
        args = (labels.to(cuda_device), lse, pz, g.to(cuda_device), q.to(cuda_device), 1.0 / t)
        apart = TU.logits_bwd(z, *args).cpu().double()
        # one rounding to the result's type, on top of fp32 arithmetic on terms of the order of the upstream gradients
        bound = zd.grad.abs() * (2.0 ** -8 if dtype == torch.bfloat16 else 0.0) + 4e-6
        assert bool(((apart - zd.grad).abs() <= bound).all())
        rest = buf.clone()
        TU.logits_bwd_(z, *args)
        assert torch.equal(z.cpu().double(), apart)
        untouched = torch.ones(buf.numel(), dtype=torch.bool)
        untouched[offset:].as_strided((T, V), (pitch, 1)).fill_(False)
        assert torch.equal(buf.cpu()[untouched], rest.cpu()[untouched])


# Logits that overflow to -inf have no probability.  A whole half tile of them (128 vocabulary rows) has a maximum of -inf and
# sums that are NaN: it takes no part in the merge, wherever it lies among the parts.  Bounds: fp32 sums, as elsewhere.
@pytest.mark.parametrize("first_row", [0, 128, 256 * 31])
@pytest.mark.parametrize("want_entropy", [False, True])
def test_half_tile_of_minus_infinity(first_row, want_entropy, cuda_device):
    T, H, V = 70, 128, 256 * 34
    hidden, weight, _, _, _ = _operands(T, H, V, seed=first_row)
    hidden = hidden.abs()
    weight[first_row:first_row + 128] = -3.0e38
    kept = torch.cat([torch.arange(first_row), torch.arange(first_row + 128, V)])
    labels = kept[torch.randint(0, kept.numel(), (T,), generator=torch.Generator().manual_seed(1))]
    lp, ent, lse, _ = ops.lmhead_fwd(hidden.to(cuda_device), weight.to(cuda_device), labels.to(cuda_device), 1.0, want_entropy)
    z = hidden.double() @ weight[kept].double().t()
    want_lse = torch.logsumexp(z, dim=1)
    label_z = (hidden.double() * weight[labels].double()).sum(dim=1)
    assert torch.allclose(lse.cpu().double(), want_lse, rtol=0, atol=1e-4)
    assert torch.allclose(lp.cpu().double(), label_z - want_lse, rtol=0, atol=1e-4)
    if want_entropy:
        p = torch.softmax(z, dim=1)
        assert torch.allclose(ent.cpu().double(), want_lse - (p * z).sum(dim=1), rtol=1e-4, atol=1e-4)


# A NaN among the logits of a token makes its log-probability, entropy and log-sum-exp NaN, also where all rows of a half tile are NaN
# and their maximum says nothing: a whole half tile, the single row of a last one, one row next to others, one next to logits that are
# -inf, every row, and a token whose hidden state is NaN.  On both kinds of tiles; tokens and calls without a NaN keep their numbers.
@pytest.mark.parametrize("T", [70, 200])
@pytest.mark.parametrize("V,first,count", [(256 * 34, 128, 128), (256 * 8 + 1, 256 * 8, 1), (256 * 8 + 133, 256 * 8 + 128, 5), (1000, 17, 1),
                                           (1000, 0, 1000)])
@pytest.mark.parametrize("want_entropy", [False, True])
def test_not_a_number_stays(T, V, first, count, want_entropy, cuda_device):
    H = 128
    hidden, weight, labels, _, _ = _operands(T, H, V, seed=V + first)
    hidden = hidden.abs()
    hidden[3] = float("nan")
    h, y = hidden.to(cuda_device), labels.to(cuda_device)

    def forward(w):
        lp, ent, lse, pz = ops.lmhead_fwd(h, w.to(cuda_device), y, 1.0, want_entropy)
        return (lp, ent, lse, pz) if want_entropy else (lp, lse)

    others = torch.arange(T, device=cuda_device) != 3
    for out in forward(weight):
        assert bool(out[~others].isnan().all()) and bool(out[others].isfinite().all())
    weight[first:first + count] = float("nan")
    assert all(bool(out.isnan().all()) for out in forward(weight))
    if first >= 128:  # and with a half tile of logits that are -inf in front of it
        weight[:128] = -3.0e38
        assert all(bool(out.isnan().all()) for out in forward(weight))


# dW of few tokens has a kernel of its own (256 x 128 tiles, steps of 32 tokens): one token, a step that is full, one short and one
# over, the last size of the rule and the first behind it; a hidden size that overhangs a tile, a last vocabulary group moved back,
# several chunks.  The accumulating call keeps the 256 x 256 tiles: the same dz panel, so both differ by fp32 sums of T products in
# another order, sqrt(T) 2^-24 = 2e-6.
@pytest.mark.parametrize("T,vc", [(1, 0), (31, 0), (32, 4096), (33, 0), (257, 4096), (768, 0), (769, 0)])
def test_weight_gradient_of_few_tokens(T, vc, cuda_device):
    H, V = 4160, 12100
    hidden, weight, labels, g, q = _operands(T, H, V, seed=T)
    labels[0] = V - 1
    if T > 2:
        g[1::3], q[1::3] = 0.0, 0.0
    h, w, y, gd, qd = (x.to(cuda_device) for x in (hidden, weight, labels, g, q))
    _, _, lse, pz = ops.lmhead_fwd(h, w, y, 1.0, True)
    want = torch.zeros(V, H, device=cuda_device)
    dh = ops.lmhead_bwd_accumulate(h, w, y, lse, pz, gd, qd, 1.0, want, vc)
    for active in (False, True):
        dh32, dw32 = ops.lmhead_bwd(h, w, y, lse, pz, gd, qd, 1.0, vc, active)
        dh16, dw16 = ops.lmhead_bwd_bf16(h, w, y, lse, pz, gd, qd, 1.0, vc, active)
        assert float((dw32 - want).norm() / want.norm()) < 1e-5
        assert torch.equal(dw16, dw32.to(torch.bfloat16)) and torch.equal(dh16, dh32)
        _close(dh16, dh.cpu(), f"dHidden T={T}")
    if T <= 33:
        _close(dw16, O.exact_fwd_bwd(hidden, weight, labels, 1.0, g, q)["d_weight"], f"dW T={T}")
    zero = torch.zeros_like(gd)
    assert not any(t.any() for t in ops.lmhead_bwd_bf16(h, w, y, lse, pz, zero, zero, 1.0, vc, True))


# Behind 96 tokens dz stays in registers, in code of its own for every 64 tokens, unless the device finds 64 and fewer or rows of hidden columns are
# short (256): the tokens with a gradient at the ends of these, more (4160) and fewer (640) hidden columns than a workgroup's share of units, the
# shortest rows (448, up to 128 tokens), a last vocabulary group moved back.  Both sides are fp32 sums of the same dz panel in
# another order, sqrt(768) 2^-24 = 2e-6.
@pytest.mark.parametrize("active", [1, 64, 65, 127, 128, 129, 193, 256, 257, 321, 385, 449, 513, 577, 640, 641, 705, 767])
@pytest.mark.parametrize("H,V", [(4160, 12100), (640, 98341), (448, 98341), (256, 196741)])
def test_weight_gradient_with_resident_dz(active, H, V, cuda_device):
    T = 97 if active < 96 else 128 if active == 127 else 768
    hidden, weight, labels, g, q = _operands(T, H, V, seed=active)
    labels[0], labels[T - 1] = V - 1, -1
    rest = torch.randperm(T, generator=torch.Generator().manual_seed(active))[active:]
    g[rest], q[rest] = 0.0, 0.0
    h, w, y, gd, qd = (x.to(cuda_device) for x in (hidden, weight, labels, g, q))
    _, _, lse, pz = ops.lmhead_fwd(h, w, y, 1.0, True)
    want = torch.zeros(V, H, device=cuda_device)
    ops.lmhead_bwd_accumulate(h, w, y, lse, pz, gd, qd, 1.0, want, 0)
    dh32, dw32 = ops.lmhead_bwd(h, w, y, lse, pz, gd, qd, 1.0, 0, True)
    dh16, dw16 = ops.lmhead_bwd_bf16(h, w, y, lse, pz, gd, qd, 1.0, 0, True)
    assert float((dw32 - want).norm() / want.norm()) < 1e-5
    assert float((dw32 - want).abs().max() / want.abs().max()) < 1e-5
    assert torch.equal(dw16, dw32.to(torch.bfloat16)) and torch.equal(dh16, dh32)


# Logits of at most 128 tokens come from 256 x 128 tiles (two steps of 32 k at H=64, the shortest): one token, a wave's 64 and one
# more, the last size of the rule and the first behind it; a vocabulary that ends inside a tile, its last group moved back (V >= 1024) or
# not, chunks of one tile, a fp32 weight with its label residual.  The forward accumulates every logit in the same order as the square
# tiles: the statistics are the bits that the same tokens get in a longer call.
@pytest.mark.parametrize("T", [1, 63, 64, 65, 127, 128, 129])
@pytest.mark.parametrize("H,V,vc,dtype", [(64, 1153, 256, torch.bfloat16), (192, 777, 0, torch.bfloat16), (320, 5001, 0, torch.bfloat16),
                                          (64, 1300, 512, torch.float32)])
def test_logits_of_few_tokens(T, H, V, vc, dtype, cuda_device):
    t = 0.7
    hidden, weight, labels, g, q = _operands(300, H, V, seed=T + V, dtype=dtype)
    labels[0], labels[T - 1] = V - 1, -1  # the vocabulary's last row; no target
    h, w, y, gd, qd = (x.to(cuda_device) for x in (hidden, weight, labels, g, q))
    longer = ops.lmhead_fwd(h, w, y, 1.0 / t, True)
    h, y, gd, qd = h[:T], y[:T], gd[:T].clone(), qd[:T]
    few = ops.lmhead_fwd(h, w, y, 1.0 / t, True)
    assert all(torch.equal(a, b[:T]) for a, b in zip(few, longer))
    if T > 2:
        gd[1::3], qd[1::3] = 0.0, 0.0
    ex = O.exact_fwd_bwd(hidden[:T], weight, labels[:T], t, gd.cpu(), qd.cpu())
    for entropy_grad in (True, False):
        if not entropy_grad:
            ex = O.exact_fwd_bwd(hidden[:T], weight, labels[:T], t, gd.cpu(), torch.zeros(T))
        for active in (False, True):
            dh, dw = ops.lmhead_bwd(h, w, y, few[2], few[3], gd, qd if entropy_grad else None, 1.0 / t, vc, active)
            _close(dh, ex["d_hidden"], f"dHidden T={T}")
            _close(dw, ex["d_weight"], f"dW T={T}")


# One sequence scored without a gradient runs on its first S - 1 positions with the ids behind the first in place of a roll: the bits of
# the differentiable call, at the shortest sequences and on both sides of the few-token rule, ids outside the vocabulary included.
@pytest.mark.parametrize("S", [1, 2, 129, 130, 300])
@pytest.mark.parametrize("temperature,ids", [(1.0, torch.int64), (0.7, torch.int32)])
def test_scoring_one_sequence(S, temperature, ids, cuda_device):
    H, V = 128, 3001
    hidden, weight, _, _, _ = _operands(S, H, V, seed=S)
    h, w = hidden.reshape(1, S, H).to(cuda_device), weight.to(cuda_device)
    tokens = torch.randint(0, V + 2, (1, S), generator=torch.Generator().manual_seed(S)).to(ids).to(cuda_device)
    scored = from_parallel_hidden_to_logprobs(h, w, tokens, 0, V, None, inference_only=True, temperature=temperature)
    assert scored.shape == (1, S - 1)
    assert torch.equal(scored, from_parallel_hidden_to_logprobs(h, w, tokens, 0, V, None, temperature=temperature).detach())


def _bwd_c_abi(h, w, y, lse, pz, g, q, vc, size, active, want_dw):
    lib = _lib.load()
    (T, H), V = h.shape, w.shape[0]
    ws = torch.empty(size, dtype=torch.uint8, device=h.device)
    dh = torch.full((T, H), float("nan"), dtype=torch.bfloat16, device=h.device)
    dw = torch.empty(V, H, device=h.device) if want_dw else None
    fn = lib.skyrl_lmhead_bwd_active_rows if active else lib.skyrl_lmhead_bwd
    st = fn(h.data_ptr(), H, w.data_ptr(), H, y.data_ptr(), lse.data_ptr(), pz.data_ptr(), g.data_ptr(), q.data_ptr(), T, H, V, 1.0,
            dh.data_ptr(), dw.data_ptr() if want_dw else None, 0, vc, ws.data_ptr(), size, torch.cuda.current_stream().cuda_stream)
    return st, dh, dw


# Scratch without room for several slabs of dHidden sums: every size down to one slab per tile, the sum of the documented terms (4 * T * H
# + 28 * T more for the gathered rows), is taken and only splits the contraction less; one byte less is refused.
@pytest.mark.parametrize("T,H,V,vc", [(300, 192, 5001, 2048), (137, 320, 5120, 5120), (700, 64, 3000, 2304)])
@pytest.mark.parametrize("active", [False, True])
@pytest.mark.parametrize("want_dw", [True, False])
def test_backward_with_less_scratch(T, H, V, vc, active, want_dw, cuda_device):
    hidden, weight, labels, g, q = _operands(T, H, V, seed=T)
    g[1::4], q[1::4] = 0.0, 0.0
    h, w, y, gd, qd = (x.to(cuda_device) for x in (hidden, weight, labels, g, q))
    _, _, lse, pz = ops.lmhead_fwd(h, w, y, 1.0, True)
    lib = _lib.load()
    query = lib.skyrl_lmhead_bwd_active_rows_workspace_bytes if active else lib.skyrl_lmhead_bwd_workspace_bytes
    full, up = query(T, H, V, vc), lambda n: -(-n // 256) * 256
    terms = [2 * H * (up(T) + 64), 4 * up(T) * up(H) + (2 * T * H if active else 0), 2 * up(T) * (vc + 64)]
    least = sum(map(up, terms + ([2 * T * H, 8 * T] + [4 * T] * 5 + [12] if active else [])))
    assert least < full
    ex = O.exact_fwd_bwd(hidden, weight, labels, 1.0, g, q)
    for size in (full, full - 1, (full + least) // 2, least):
        st, dh, dw = _bwd_c_abi(h, w, y, lse, pz, gd, qd, vc, size, active, want_dw)
        assert st == 0, (size, least, full)
        _close(dh, ex["d_hidden"], f"dHidden, {size} bytes")
        if want_dw:
            _close(dw, ex["d_weight"], f"dW, {size} bytes")
    assert _bwd_c_abi(h, w, y, lse, pz, gd, qd, vc, least - 1, active, want_dw)[0] == ERR_WORKSPACE


# Scratch sized once, for the longest call, serves the shorter ones: with a chunk that is given, and with the library's own.
@pytest.mark.parametrize("T,longest,H,V,vc", [(3072, 3584, 3584, 8192, 4096), (5000, 16384, 512, 152064, 0)])
@pytest.mark.parametrize("active", [False, True])
def test_backward_scratch_of_a_longer_call(T, longest, H, V, vc, active, cuda_device):
    gen = torch.Generator(device=cuda_device).manual_seed(T)
    h = torch.randn(T, H, generator=gen, device=cuda_device).to(torch.bfloat16)
    w = (torch.randn(V, H, generator=gen, device=cuda_device) * 3 / H**0.5).to(torch.bfloat16)
    y = torch.randint(0, V, (T,), generator=gen, device=cuda_device)
    g, q = (torch.randn(T, generator=gen, device=cuda_device) for _ in range(2))
    _, _, lse, pz = ops.lmhead_fwd(h, w, y, 1.0, True)
    lib = _lib.load()
    query = lib.skyrl_lmhead_bwd_active_rows_workspace_bytes if active else lib.skyrl_lmhead_bwd_workspace_bytes
    st, want, _ = _bwd_c_abi(h, w, y, lse, pz, g, q, vc, query(T, H, V, vc), active, False)
    assert st == 0
    st, got, _ = _bwd_c_abi(h, w, y, lse, pz, g, q, vc, query(longest, H, V, vc), active, False)
    assert st == 0
    # The fp32 sums are added in another order, 1e-5 of a value at most: up to 1e-5 / 2^-8 of the values round to the neighbouring bf16,
    # 2^-8 away, 2e-4 in the 2-norm.
    assert float((got.float() - want.float()).norm() / want.float().norm()) < 1e-3


# The draft loss's backward in scratch of the documented terms (stacked rows, one dHidden's sums, the panel), which leave no room for the
# inputs of the listed tokens, and in scratch that was sized for a longer call; below those terms it is refused.
@pytest.mark.parametrize("T,H,V,vc", [(300, 192, 5001, 2048), (137, 320, 5120, 5120), (700, 64, 3000, 512), (300, 128, 700, 256)])
def test_draft_loss_backward_with_less_scratch(T, H, V, vc, cuda_device):
    student, weight, _, g, _ = _operands(T, H, V, seed=T)
    teacher = _operands(T, H, V, seed=T + 1)[0]
    g[1::4] = 0.0
    hs, ht, w, gd = (x.to(cuda_device) for x in (student, teacher, weight, g))
    _, lse_s, lse_t = softce_fwd(hs, ht, w, T, 1, 1.0)
    lib = _lib.load()
    up, Tp = lambda n, m=256: -(-n // m) * m, -(-T // 128) * 128
    terms = [4 * Tp * H, 4 * up(T) * up(H), 2 * Tp * (vc + 64)]
    least = sum(map(up, terms + ([] if V >= 1024 else [2 * H * (up(V) + 64)])))
    if vc == 256:  # no column to spare
        least += sum(map(up, [4 * T] * 4 + [12]))
    full = lib.skyrl_softce_bwd_workspace_bytes(T, H, V, vc)
    sizes = {full, max(full - 1, least), (full + least) // 2, least, lib.skyrl_softce_bwd_workspace_bytes(2 * T, H, V, vc)}
    want = softce_bwd(hs, ht, w, lse_s, lse_t, gd, T, 1, 1.0, vc)
    hd = student.double().requires_grad_(True)
    ls, lt = hd @ weight.double().T, torch.roll(teacher, -1, 0).double() @ weight.double().T
    (-(lt.softmax(-1) * ls.log_softmax(-1)).sum(-1) * g.double()).sum().backward()
    _close(want, hd.grad, "d student")

    def call(size):
        ws = torch.empty(size, dtype=torch.uint8, device=cuda_device)
        d = torch.full_like(hs, float("nan"))
        st = lib.skyrl_softce_bwd(hs.data_ptr(), H, ht.data_ptr(), H, w.data_ptr(), H, lse_s.data_ptr(), lse_t.data_ptr(), gd.data_ptr(), T,
                                  T, 1, H, V, 1.0, d.data_ptr(), vc, ws.data_ptr(), size, torch.cuda.current_stream().cuda_stream)
        return st, d

    for size in sizes:
        st, d = call(size)
        assert st == 0, (size, least, full)
        _close(d, hd.grad, f"d student, {size} bytes")
    assert call(least // 2)[0] == ERR_WORKSPACE and (vc > 256 or call(least - 1)[0] == ERR_WORKSPACE)


# The last token tile is made narrower where it holds no more than 128 or 192 tokens.  A token's values do not depend on the width of its
# tile: the last tokens of a call are compared, bit for bit, with those of a longer call.  (These vocabularies give no more than 128 tiles,
# which the longer call makes as short ones; test_shapes_against_square_tiles compares with square ones.)
@pytest.mark.parametrize("T", [257, 319, 320, 384, 385, 447, 448, 449, 513])
@pytest.mark.parametrize("H,V", [(64, 1153), (128, 5001), (192, 777), (320, 2304)])
def test_last_tokens_in_a_narrow_tile(T, H, V, cuda_device):
    t = 0.8
    hidden, weight, labels, g, q = _operands(768, H, V, seed=T + H)
    h, w, y, gd, qd = (x.to(cuda_device) for x in (hidden, weight, labels, g, q))
    long = ops.lmhead_fwd(h, w, y, 1.0 / t, True)
    short = ops.lmhead_fwd(h[:T], w, y[:T], 1.0 / t, True)
    for a, b in zip(short, long):
        assert torch.equal(a, b[:T])
    assert torch.equal(ops.lmhead_fwd(h[:T], w, y[:T], 1.0 / t, False)[0], ops.lmhead_fwd(h, w, y, 1.0 / t, False)[0][:T])
    lse, pz = short[2], short[3]
    ex = O.exact_fwd_bwd(hidden[:T], weight, labels[:T], t, g[:T], q[:T])
    dh, dw = ops.lmhead_bwd(h[:T], w, y[:T], lse, pz, gd[:T], qd[:T], 1.0 / t, 0)
    _close(dh, ex["d_hidden"], f"dHidden T={T}")
    _close(dw, ex["d_weight"], f"dW T={T}")
    dropped = gd.clone()  # the same tokens, found by the compaction among others
    dropped[T:], qd[T:] = 0.0, 0.0
    dh2, dw2 = ops.lmhead_bwd(h, w, y, long[2], long[3], dropped, qd, 1.0 / t, 0, True)
    _close(dh2[:T], ex["d_hidden"], f"dHidden of {T} active tokens")
    _close(dw2, ex["d_weight"], f"dW of {T} active tokens")
    assert not dh2[T:].any()
    for k in (5, 200):
        for a, b in zip(topk_logits_from_hidden(h[:T], w, k), topk_logits_from_hidden(h, w, k)):
            assert torch.equal(a, b[:T])


# The merge takes eight or ten parts (128 vocabulary rows each) a step, by how many there are per stream: both sides of every line of that
# rule.  fp32 statistics of bf16 products: 1e-5 relative covers their summation orders.
@pytest.mark.parametrize("streams", [1, 8, 10, 16, 20])
@pytest.mark.parametrize("more", [0, 1])
def test_parts_of_the_forward_merge(streams, more, cuda_device):
    T, H, V = 17, 64, streams * 64 * 128 + more
    hidden, weight, labels, _, _ = _operands(T, H, V, seed=V)
    labels[:3] = torch.tensor([V - 1, 0, V // 2])
    ex = O.exact_fwd_bwd(hidden, weight, labels, 0.9)
    lp, ent, *_ = ops.lmhead_fwd(hidden.to(cuda_device), weight.to(cuda_device), labels.to(cuda_device), 1.0 / 0.9, True)
    torch.testing.assert_close(lp.double().cpu(), ex["logprobs"], rtol=1e-5, atol=1e-5)
    torch.testing.assert_close(ent.double().cpu(), ex["entropy"], rtol=1e-5, atol=1e-5)


# The tiles of a last round that fills no more than half of the CUs are made as short ones, the rest as square ones: 133 tile rows give
# none for one token tile (T=40: half tiles, 137: medium ones, 256: square ones), 256 square and 10 short ones for two, and none for three,
# whose values are the measure, bit for bit.  The vocabulary ends in the lower half of its last tile, at its middle, and in the upper half.
@pytest.mark.parametrize("V", [33900, 33920, 34001])
@pytest.mark.parametrize("T", [40, 137, 256, 300, 512])
def test_last_round_in_short_tiles(T, V, cuda_device):
    H, t = 128, 0.8
    hidden, weight, labels, g, q = _operands(768, H, V, seed=V)
    labels[:4] = torch.tensor([V - 1, 132 * 256, 132 * 256 + 107, 0])
    h, w, y, gd, qd = (x.to(cuda_device) for x in (hidden, weight, labels, g, q))
    for want_entropy in (False, True):
        long, short = ops.lmhead_fwd(h, w, y, 1.0 / t, want_entropy), ops.lmhead_fwd(h[:T], w, y[:T], 1.0 / t, want_entropy)
        for a, b in zip(short, long):
            assert torch.equal(a, b[:T])
    for a, b in zip(topk_logits_from_hidden(h[:T], w, 5), topk_logits_from_hidden(h, w, 5)):
        assert torch.equal(a, b[:T])
    # d_hidden of the same tokens, alone and found by the compaction, with the whole vocabulary in one chunk and in two
    gd[T:], qd[T:] = 0.0, 0.0
    ex = O.exact_fwd_bwd(hidden[:T], weight, labels[:T], t, g[:T], q[:T])
    for vc in (0, 17408):
        dh, dw = ops.lmhead_bwd(h[:T], w, y[:T], short[2], short[3], gd[:T], qd[:T], 1.0 / t, vc)
        _close(dh, ex["d_hidden"], f"dHidden T={T} chunk={vc}")
        _close(dw, ex["d_weight"], f"dW T={T} chunk={vc}")
        dh, dw = ops.lmhead_bwd(h, w, y, long[2], long[3], gd, qd, 1.0 / t, vc, True)
        _close(dh[:T], ex["d_hidden"], f"dHidden of {T} active tokens, chunk={vc}")
        _close(dw, ex["d_weight"], f"dW of {T} active tokens, chunk={vc}")


# The draft loss's masked mean: the mask's own sum counts, once per value where it is broadcast over the sequences, and is at least one.
@pytest.mark.parametrize("shape", [(3, 41), (1, 41)])
@pytest.mark.parametrize("share", [0.0, 0.01, 0.6])
def test_masked_mean_of_the_draft_loss(shape, share, cuda_device):
    B, S, H, V = 3, 41, 64, 1500
    hidden, weight, *_ = _operands(2 * B * S, H, V, seed=S)
    student, teacher = (x.reshape(B, S, H).to(cuda_device) for x in hidden.split(B * S))
    mask = (torch.rand(shape, generator=torch.Generator().manual_seed(7)) < share).to(cuda_device)
    up = torch.tensor(0.7, device=cuda_device)
    for loss_of, per_token_of in (
            (lambda s: draft_soft_ce_from_hidden(s, teacher, weight.to(cuda_device), mask),
             lambda s: soft_ce_from_hidden(s, teacher, weight.to(cuda_device), shift=1)),
            (lambda s: draft_soft_ce_topk_from_hidden(s, teacher, weight.to(cuda_device), mask, 9, roll_shift=1),
             lambda s: soft_ce_topk_from_hidden(s, teacher, weight.to(cuda_device), 9, shift=1))):
        s, r = (student.clone().requires_grad_(True) for _ in range(2))
        loss, per_token = loss_of(s), per_token_of(r)
        want = (per_token.double() * mask).sum() / mask.double().sum().clamp(min=1.0)
        assert loss.shape == () and abs(float(loss.detach()) - float(want.detach())) <= 1e-6 * max(1.0, abs(float(want.detach())))
        (loss * up).backward()
        (want * up).backward()  # the upstream per token differs in fp32 roundings only, which d_hidden's bf16 rounding may turn into an ulp
        assert torch.allclose(s.grad.float(), r.grad.float(), rtol=2**-7, atol=1e-7)


@pytest.mark.parametrize("shape", [(2, 41), (1, 41)])
@pytest.mark.parametrize("topk", [False, True])
def test_draft_loss_scaled_in_place(shape, topk, cuda_device):
    B, S, H, V = 2, 41, 64, 1500
    hidden, weight, *_ = _operands(2 * B * S, H, V, seed=S)
    student, teacher = (x.reshape(B, S, H).to(cuda_device) for x in hidden.split(B * S))
    mask, w = torch.ones(shape, device=cuda_device), weight.to(cuda_device)
    loss_of = (lambda s: draft_soft_ce_topk_from_hidden(s, teacher, w, mask, 9)) if topk else (lambda s: draft_soft_ce_from_hidden(s, teacher, w, mask))
    s, r = (student.clone().requires_grad_(True) for _ in range(2))
    loss, whole = loss_of(s), loss_of(r)
    loss *= 0.5
    loss.backward()
    whole.backward()
    assert torch.equal(loss.detach(), 0.5 * whole.detach()) and torch.equal(s.grad, 0.5 * r.grad)  # halves are exact


# Square tiles are the measure of all other shapes, bit for bit and behind the first k-tiles too (three, four and five of them): 50 tile rows
# make 150 tiles of 768 tokens, more than half of the CUs and no remainder, so all square; for one and two token tiles no more than 128,
# so all short or, where the last column is narrow, that; and for three a last column of its own width beside square ones.  The vocabulary ends
# in the lower half of its last tile, at its middle, and in the upper half.  Top-k: 1024 tokens of 128 tile rows are two chunks of 256 tiles.
@pytest.mark.parametrize("H", [192, 256, 320])
@pytest.mark.parametrize("rest", [100, 128, 200])
def test_shapes_against_square_tiles(H, rest, cuda_device):
    V, wide = 49 * 256 + rest, 127 * 256 + rest
    hidden, weight, labels, *_ = _operands(1024, H, wide, seed=H + rest)
    h, w, y = hidden.to(cuda_device), weight.to(cuda_device), labels.remainder(V).to(cuda_device)
    whole = [ops.lmhead_fwd(h[:768], w[:V], y[:768], 1.25, ent) for ent in (False, True)]
    first = [topk_logits_from_hidden(h, w, k) for k in (5, 200)]
    for T in (137, 256, 300, 512, 513, 640, 641, 700, 704):
        for ent in (False, True):
            for a, b in zip(ops.lmhead_fwd(h[:T], w[:V], y[:T], 1.25, ent), whole[ent]):
                assert torch.equal(a, b[:T]), (T, ent)
        for k, want in zip((5, 200), first):
            for a, b in zip(topk_logits_from_hidden(h[:T], w, k), want):
                assert torch.equal(a, b[:T]), (T, k)
    # the draft loss: two rows per token
    ht = h.flip(0)[:384].contiguous()
    pairs = softce_fwd(h[:384], ht, w[:V], 384, 0, 1.25)
    for T in (69, 128, 150, 256, 257, 320, 321, 340, 352):
        for a, b in zip(softce_fwd(h[:T], ht[:T], w[:V], T, 0, 1.25), pairs):
            assert torch.equal(a, b[:T]), T


# The draft loss stacks a student's and a teacher's row per token, so its last tile is made narrower where it holds no more than 64 or 96
# tokens, and a last round in short tiles.  Values do not depend on the tile's shape: the first tokens of a longer call are the measure, bit
# for bit (square tiles with 133 tile rows, V=34001; short ones with fewer).
@pytest.mark.parametrize("T", [1, 16, 17, 64, 65, 96, 97, 128, 129, 208, 300])
@pytest.mark.parametrize("H,V", [(64, 1153), (320, 5001), (128, 34001)])
def test_last_tokens_of_the_draft_loss(T, H, V, cuda_device):
    hidden, weight, _, g, _ = _operands(384, H, V, seed=T + H)
    teacher = torch.randn(384, H, generator=torch.Generator().manual_seed(V)).to(torch.bfloat16)
    h, ht, w, gd = (x.to(cuda_device) for x in (hidden, teacher, weight, g))
    long = softce_fwd(h, ht, w, 384, 0, 1.0)
    short = softce_fwd(h[:T], ht[:T], w, T, 0, 1.0)
    for a, b in zip(short, long):
        assert torch.equal(a, b[:T])
    zs, zt = hidden[:T].double() @ weight.double().t(), teacher[:T].double() @ weight.double().t()
    want = (g[:T].double()[:, None] * (zs.softmax(-1) - zt.softmax(-1))) @ weight.double()
    gd[T:] = 0.0
    for vc in (0, 1024):
        _close(softce_bwd(h[:T], ht[:T], w, short[1], short[2], gd[:T], T, 0, 1.0, vc), want, f"d student T={T}")
        d = softce_bwd(h, ht, w, long[1], long[2], gd, 384, 0, 1.0, vc)  # the same tokens, found by the compaction among others
        _close(d[:T], want, f"d student of {T} active tokens")
        assert not d[T:].any()
