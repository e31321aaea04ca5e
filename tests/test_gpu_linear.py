"""
nsmoe_linear (nanospeaker_amd/csrc/linear.hip) against the same product in 64 bits: x W and
x W + resid with one rounding of the fp32 sum, at the edges of its row tiles (32 to 128 rows)
and of the row counts that choose them, of a wave's 48, 32 and 16 columns and of a pass of 576,
and through the attention sublayer with operands the kernel cannot read in place; and the
packed weights it reads, across streams, captures and updates.
"""

import pytest
import torch

pytestmark = pytest.mark.gpu

pytest.importorskip("nanospeaker_amd.moe_kernel")
from nanospeaker_amd import _native as nat  # noqa: E402
from nanospeaker_amd.decoder import (Attention, DecoderConfig, Rotary, linear,  # noqa: E402
                                     pack_linear)
from nanospeaker_amd.moe_kernel import PACKS  # noqa: E402

DEV = "cuda"


def _operands(M, K, N, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(M, K, generator=g).to(dtype).to(DEV)
    w = (torch.randn(K, N, generator=g) * 0.05).to(dtype).to(DEV)
    r = torch.randn(M, N, generator=g).to(dtype).to(DEV)
    return x, w, r


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,K,N", [
    (1, 576, 960), (31, 576, 960), (33, 576, 576), (127, 64, 16), (129, 32, 48), (300, 544, 592),
    (4097, 576, 960), (8193, 576, 576), (12289, 576, 960), (16385, 576, 576), (28800, 576, 576), (28673, 96, 976), (500, 576, 1152),
    (77, 320, 1328)])
def test_linear_against_64_bits(M, K, N, dtype):
    """A result is one rounding of an fp32 sum: within the dtype's unit roundoff (2^-8 for
    bf16's 8 significant bits, 2^-11 for fp16's 11) of the exact one plus the sum's own error, K
    terms of 2^-24 of their magnitude sum.  In place (out = resid) and without a residual."""
    x, w, r = _operands(M, K, N, dtype, M + N)
    print(f"[linear] {M} x {K} x {N} {dtype}", flush=True)
    wp = pack_linear(w)
    step = 2.0 ** -8 if dtype is torch.bfloat16 else 2.0 ** -11
    xd, wd = x.double(), w.double()
    mags = xd.abs() @ wd.abs()
    for resid in (None, r):
        ref = xd @ wd + (0 if resid is None else r.double())
        bound = ref.abs() * step * 1.01 + (mags + (0 if resid is None else r.double().abs())) * (
            K * 2.0 ** -24) + 1e-7
        got = linear(x, wp, N, resid)
        assert ((got.double() - ref).abs() <= bound).all()
    acc = r.clone()
    out = linear(x, wp, N, acc, acc)
    assert out.data_ptr() == acc.data_ptr() and torch.equal(out, got)


def test_linear_rejects_what_it_does_not_take():
    x, w, r = _operands(8, 64, 32, torch.bfloat16, 0)
    wp = pack_linear(w)
    args = lambda k=64, n=32, out=r: (nat.BF16, x.data_ptr(), 8, k, n, wp.data_ptr(), None,
                                      out.data_ptr(), None)
    for bad in (args(k=48), args(k=608), args(n=24), args(out=r.view(-1)[1:])):
        assert nat.lib().nsmoe_linear(*bad) == 1
    assert nat.lib().nsmoe_linear(nat.F32, *args()[1:]) == 1
    assert nat.lib().nsmoe_linear(nat.BF16, None, 0, 64, 32, None, None, None, None) == 0


@pytest.mark.parametrize("d_model", [576, 584])
def test_attention_sublayer_operands(d_model):
    """forward_residual with strided, misaligned and in-place operands, and with a d_model the
    kernel does not take (584: torch products), all equal to the plain call; an in-place
    weight update is seen."""
    torch.manual_seed(0)
    cfg = DecoderConfig(d_model=d_model)
    att = Attention(cfg, Rotary(64, cfg.rope_base), None).to(DEV, torch.bfloat16).eval()
    x = torch.randn(2, 70, d_model, device=DEV, dtype=torch.bfloat16)
    z = torch.randn_like(x)
    odd = lambda t: torch.cat((t.new_zeros(1), t.reshape(-1)))[1:].view(t.shape)
    with torch.no_grad():
        ref = att.forward_residual(x, z)
        assert torch.equal(att.forward_residual(x, z.transpose(0, 1).contiguous().transpose(0, 1)),
                           ref)
        assert torch.equal(att.forward_residual(odd(x), odd(z)), ref)
        for own in (x.clone(), odd(x)):
            got = att.forward_residual(own, z, inplace=True)
            assert got.data_ptr() == own.data_ptr() and torch.equal(got, ref)
        att.W_O.mul_(2.0)
        assert not torch.equal(att.forward_residual(x, z), ref)


def test_attention_refuses_a_residual_that_does_not_fit():
    """A residual of other rows, another width, dtype or device than the layer's output is
    refused on the host, in place or not; W_O in another dtype than the tokens is refused by
    the plain forward, as a torch product of mixed operands is."""
    cfg = DecoderConfig()
    att = Attention(cfg, Rotary(64, cfg.rope_base), None).to(DEV, torch.bfloat16).eval()
    z = torch.randn(2, 70, 576, device=DEV, dtype=torch.bfloat16)
    with torch.no_grad():
        for x in (z[:, :69].contiguous(), z[:1], torch.cat((z, z), dim=-1), z[..., :64].contiguous(),
                  z.cpu()):
            for inplace in (False, True):
                with pytest.raises(RuntimeError):
                    att.forward_residual(x, z, inplace=inplace)
        att.W_O.data = att.W_O.data.float()
        with pytest.raises(RuntimeError):
            att(z)


def test_plain_attention_reads_the_current_output_weight():
    """forward() on the kernel path is the attention's output times W_O by torch's product,
    bit for bit, also after a write through `.data`."""
    torch.manual_seed(1)
    cfg = DecoderConfig()
    att = Attention(cfg, Rotary(64, cfg.rope_base), None).to(DEV, torch.bfloat16).eval()
    z = torch.randn(2, 70, 576, device=DEV, dtype=torch.bfloat16)
    with torch.no_grad():
        for _ in range(2):
            o = att._kernel_attention(z).view(2, 70, -1)
            assert torch.equal(att(z), o @ att.W_O)
            att.W_O.data.mul_(2.0)


def _attention_and_inputs(rotary=None):
    cfg = DecoderConfig()
    att = Attention(cfg, rotary or Rotary(64, cfg.rope_base), None).to(DEV, torch.bfloat16).eval()
    g = torch.Generator().manual_seed(3)
    x, z = (torch.randn(2, 70, 576, generator=g).to(DEV, torch.bfloat16) for _ in range(2))
    return att, x, z


def test_projection_packs_on_another_stream():
    """A pack made behind long work on one stream is waited for by a call on another one."""
    att, x, z = _attention_and_inputs()
    with torch.no_grad():
        ref = att.forward_residual(x, z)
        PACKS.clear()
        torch.cuda.synchronize()
        one, two = torch.cuda.Stream(), torch.cuda.Stream()
        with torch.cuda.stream(one):
            torch.cuda._sleep(20_000_000)
            first = att.forward_residual(x, z)
        with torch.cuda.stream(two):
            second = att.forward_residual(x, z)
        torch.cuda.synchronize()
        assert torch.equal(first, ref) and torch.equal(second, ref)


def _capture(fn):
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        out = fn()
    return graph, out


@pytest.mark.parametrize("warm", [True, False])
def test_captured_projections_follow_the_weights(warm):
    """A captured sublayer packs in its graph, whether its weights' packs were kept before or
    not: every replay has the weights of that moment, and eager calls after a capture (with no
    replay yet) and between replays have theirs."""
    att, x, z = _attention_and_inputs()
    other, _, _ = _attention_and_inputs(att.rotary)
    with torch.no_grad():
        other.forward_residual(x, z)  # the rotary tables
        if warm:
            att.forward_residual(x, z)
        graph, out = _capture(lambda: att.forward_residual(x, z))
        for step in range(4):
            eager = att.forward_residual(x, z)
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, eager), step
            for w in (att.W_O, att.W_k):
                w.mul_(1.5)


def test_captured_projections_share_kept_packs():
    """With share_with_graphs a capture reads the kept packs, which stay until clear(): a
    replay has the new weights after refresh(), also when the layer object itself is gone."""
    att, x, z = _attention_and_inputs()
    weights = (att.W_q, att.W_k, att.W_v, att.W_O)
    gains_and_tables = (att.q_norm, att.k_norm, att.rotary)
    with torch.no_grad():
        att.forward_residual(x, z)
        PACKS.share_with_graphs = True
        try:
            graph, out = _capture(lambda: att.forward_residual(x, z))
        finally:
            PACKS.share_with_graphs = False
        for step in range(3):
            ref = att.forward_residual(x, z)
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, ref), step
            for w in weights:
                w.mul_(1.25)
            assert PACKS.refresh() >= 2
        ref = att.forward_residual(x, z)
        del att
        spare = [torch.full((576 * 960,), float("nan"), device=DEV, dtype=torch.bfloat16)
                 for _ in range(8)]
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, ref) and len(spare) == 8 and gains_and_tables
    PACKS.clear()


@pytest.mark.parametrize("M", [16385, 20480, 20481, 24577, 28673, 32769, 41000, 50000])
def test_linear_row_tiles_of_long_calls(M):
    """Row counts that choose tiles of 80, 96, 112 and 128 rows (256 CUs: one round, then two),
    whole and ragged at the end, against the same rows in calls of at most 8,000 (32-row tiles):
    a row's products are summed in the same order whatever its tile, so the bits are equal."""
    x, w, r = _operands(M, 96, 592, torch.bfloat16, M)
    wp = pack_linear(w)
    print(f"[linear] {M} rows", flush=True)
    for resid in (None, r):
        got = linear(x, wp, 592, resid)
        for s in range(0, M, 8000):
            part = slice(s, min(M, s + 8000))
            want = linear(x[part], wp, 592, None if resid is None else resid[part].contiguous())
            assert torch.equal(got[part], want), s
