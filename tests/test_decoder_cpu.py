"""
The decoder harness around the MoE block (nanospeaker_amd/decoder.py) on the CPU: the
blocked sliding-window attention equals one SDPA call under the full band mask, the
rotary embedding is a rotation whose attention logits depend only on the offset, the
window / global layer pattern is the reference's (nanospeaker.py:102-114), and a small
decoder runs end to end on the block's eager path.
"""

import pytest
import torch
import torch.nn.functional as F

from nanospeaker_amd.decoder import (Decoder, DecoderConfig, Rotary, band_attention)


@pytest.mark.parametrize("T,w,hq,hk", [(64, 16, 4, 2), (50, 16, 3, 3), (17, 8, 6, 2),
                                       (8, 16, 2, 1)])
def test_band_attention_equals_full_band_mask(T, w, hq, hk):
    g = torch.Generator().manual_seed(T + w)
    q = torch.randn(2, hq, T, 8, generator=g, dtype=torch.float64)
    k = torch.randn(2, hk, T, 8, generator=g, dtype=torch.float64)
    v = torch.randn(2, hk, T, 8, generator=g, dtype=torch.float64)
    pos = torch.arange(T)
    allowed = (pos[None, :] <= pos[:, None]) & (pos[:, None] - pos[None, :] < w)
    ref = F.scaled_dot_product_attention(q, k, v, attn_mask=allowed, enable_gqa=hq != hk)
    got = band_attention(q, k, v, w) if w < T else None
    if got is not None:
        torch.testing.assert_close(got, ref, rtol=1e-12, atol=1e-12)


def test_rotary_is_a_rotation_with_relative_logits():
    rot = Rotary(16, 500_000.0)
    g = torch.Generator().manual_seed(1)
    q = torch.randn(1, 1, 40, 16, generator=g, dtype=torch.float64)
    k = torch.randn(1, 1, 40, 16, generator=g, dtype=torch.float64)
    # the same vector at every position: q_m . k_n must depend on m - n only (the angles
    # are formed in fp32, as the reference forms them: agreement to fp32 rounding)
    qs, ks = q[:, :, :1].expand(-1, -1, 40, -1), k[:, :, :1].expand(-1, -1, 40, -1)
    s = rot(qs)[0, 0] @ rot(ks)[0, 0].t()
    for off in (0, 3, 17):
        d = torch.diagonal(s, -off)
        torch.testing.assert_close(d, d[:1].expand_as(d), rtol=1e-6, atol=1e-6)
    # norms preserved (a rotation), and position 0 unchanged
    torch.testing.assert_close(rot(q).norm(dim=-1), q.norm(dim=-1), rtol=1e-6, atol=1e-6)
    torch.testing.assert_close(rot(q)[..., 0, :], q[..., 0, :])
    # against complex multiplication: plane j = (x_j, x_{j+8}) turned by m * base^(-j/8)
    m, j = 5, 3
    theta = m * 500_000.0 ** (-2 * j / 16)
    z = complex(q[0, 0, m, j], q[0, 0, m, j + 8]) * complex(torch.cos(torch.tensor(theta)),
                                                          torch.sin(torch.tensor(theta)))
    r = rot(q)[0, 0, m]
    assert abs(float(r[j]) - z.real) < 1e-6 and abs(float(r[j + 8]) - z.imag) < 1e-6


def test_layer_windows_follow_global_every():
    cfg = DecoderConfig()
    wins = [cfg.layer_window(i) for i in range(cfg.n_layers)]
    assert wins.count(None) == 5 and all(wins[i] is None for i in range(0, 20, 4))
    assert all(w == 512 for i, w in enumerate(wins) if i % 4)


def test_small_decoder_runs_on_the_eager_block_path():
    torch.manual_seed(0)
    cfg = DecoderConfig(vocab_size=64, d_model=32, n_layers=4, n_heads=4, n_kv_heads=2,
                        d_head=8, n_experts=8, n_shared=1, top_k=2, d_expert=16, window=8,
                        global_every=2)
    m = Decoder(cfg).eval()
    idx = torch.randint(0, 64, (2, 20))
    with torch.no_grad():
        logits = m(idx)
    assert logits.shape == (2, 20, 64) and torch.isfinite(logits).all()
    # causality: changing a later token leaves earlier logits unchanged
    idx2 = idx.clone()
    idx2[:, 15] = (idx2[:, 15] + 1) % 64
    with torch.no_grad():
        logits2 = m(idx2)
    torch.testing.assert_close(logits2[:, :15], logits[:, :15], rtol=0, atol=0)
    assert not torch.equal(logits2[:, 15:], logits[:, 15:])


def test_decoder_loss_is_the_reference_next_token_cross_entropy():
    """forward(idx, targets) (nanospeaker.py:241-250): position t predicts token t + 1,
    mean cross-entropy of the tied head's logits; on the CPU head.linear_cross_entropy is
    F.cross_entropy of the materialised fp32 logits, exactly."""
    torch.manual_seed(0)
    cfg = DecoderConfig(n_layers=1, vocab_size=64, window=None, global_every=None)
    model = Decoder(cfg, kernel=False).eval()
    idx = torch.randint(0, 64, (2, 10))
    loss, aux = model(idx, targets=idx)
    with torch.no_grad():
        x, _ = model.trunk(idx)
        ref = F.cross_entropy((x[:, :-1].reshape(-1, 576) @ model.embed.weight.t()).float(),
                              idx[:, 1:].reshape(-1))
    torch.testing.assert_close(loss, ref, rtol=0, atol=0)
    assert aux.shape == ()


def test_trunk_balance_loss_is_the_promoted_sum_of_the_blocks():
    """trunk's aux equals the reference's fp32 accumulation aux + a (nanospeaker.py:220-230)
    of each block's balance loss under type promotion, for a 16-bit model in training (a
    16-bit loss per block) and in eval (the blocks' zeros)."""
    torch.manual_seed(1)
    cfg = DecoderConfig(n_layers=3, vocab_size=64, window=None, global_every=None)
    model = Decoder(cfg, kernel=False).to(torch.bfloat16)
    idx = torch.randint(0, 64, (2, 12))
    for train in (True, False):
        model.train(train)
        with torch.no_grad():
            _, aux = model.trunk(idx)
        ref = torch.zeros((), dtype=torch.float32)
        for blk in model.blocks:
            ref = ref + blk.ffn.aux_loss
        assert aux.dtype == torch.float32
        assert torch.equal(aux, ref), (train, aux, ref)
        assert (float(aux) != 0.0) == train


def test_linear_refuses_operands_that_do_not_fit():
    """The projection kernel reads and writes through the sizes it is given, so the wrapper
    refuses, before any launch, an addend or output of other rows, columns, dtype or layout,
    a width the packed weights do not have, and host tensors."""
    from nanospeaker_amd.decoder import linear, pack_linear

    x, w = torch.zeros(4, 64, dtype=torch.bfloat16), torch.zeros(64, 32, dtype=torch.bfloat16)
    wp, ok = pack_linear(w), torch.zeros(4, 32, dtype=torch.bfloat16)
    for args in ((x, wp, 48), (x, wp, 33), (x[:, :32], wp, 32), (x, wp, 32, ok[:3]),
                 (x, wp, 32, ok[:, :16]), (x, wp, 32, ok.float()), (x, wp, 32, ok[:1]),
                 (x, wp, 32, torch.zeros(32, 4, dtype=torch.bfloat16).t()),
                 (x, wp, 32, ok, ok[:3]), (x, wp, 32)):
        with pytest.raises(RuntimeError, match="linear"):
            linear(*args)


def test_attention_packs_survive_a_module_saved_without_them():
    """A module object pickled before the weights' packed copies were kept has no `_packs`."""
    from nanospeaker_amd.decoder import Attention

    cfg = DecoderConfig(d_model=64, n_heads=1, n_kv_heads=1)
    att = Attention(cfg, Rotary(64, cfg.rope_base), None)
    del att._packs
    assert att._packed("o", torch.bfloat16, att.W_O).shape == (4, 2, 4, 16, 8)
    assert len(att._packs) == 1


def _kernel_path_on_the_cpu(monkeypatch, att, o):
    """The module's kernel path with its launches replaced: the attention's output is `o`,
    and the projection kernel is a torch product by the unpacked weights."""
    from nanospeaker_amd import decoder as D

    def linear(x, w_packed, n, resid=None, out=None):
        nb, kb = w_packed.shape[:2]
        y = x @ w_packed.permute(1, 2, 4, 0, 3).reshape(kb * 32, nb * 16)
        y = y if resid is None else y + resid
        return y if out is None else out.copy_(y)

    monkeypatch.setattr(D, "linear", linear)
    monkeypatch.setattr(att, "use_kernel", lambda z: True)
    monkeypatch.setattr(att, "_kernel_attention", lambda z: o)


def _small_attention():
    from nanospeaker_amd.decoder import Attention

    cfg = DecoderConfig(d_model=64, n_heads=1, n_kv_heads=1)
    return Attention(cfg, Rotary(64, cfg.rope_base), None).eval()


def test_plain_attention_reads_the_current_output_weight(monkeypatch):
    """Attention.forward multiplies by W_O as it is at the call, also after writes that the
    version counter does not see and after the parameter was replaced at the same address."""
    att, o, z = _small_attention(), torch.randn(6, 64), torch.zeros(2, 3, 64)
    _kernel_path_on_the_cpu(monkeypatch, att, o)
    with torch.no_grad():
        for _ in range(2):
            assert torch.equal(att(z), o.view(2, 3, 64) @ att.W_O)
            att.W_O.data.mul_(2.0)
            assert torch.equal(att(z), o.view(2, 3, 64) @ att.W_O)
            att.W_O.data.add_(1.0)
            att.W_O = torch.nn.Parameter(att.W_O.data)


def _unpacked(w):
    return w.permute(1, 2, 4, 0, 3).reshape(w.shape[1] * 32, w.shape[0] * 16)


def test_projection_packs_follow_their_parameters():
    """A kept pack belongs to the parameter objects: it is reused while they are unchanged,
    and made anew after an in-place update, and for another parameter at the same address and
    version.  After a write through `.data` PACKS.clear() drops it and PACKS.refresh() rewrites
    it in its place."""
    from nanospeaker_amd.moe_kernel import PACKS

    att, dt = _small_attention(), torch.float32
    packed = lambda: att._packed("o", dt, att.W_O)
    first = packed()
    assert torch.equal(_unpacked(first), att.W_O)
    assert packed() is first
    with torch.no_grad():
        att.W_O.mul_(2.0)
    second = packed()
    assert torch.equal(_unpacked(second), att.W_O) and not torch.equal(first, second)
    att.W_O.data.add_(1.0)
    att.W_O = torch.nn.Parameter(att.W_O.data)
    third = packed()
    assert torch.equal(_unpacked(third), att.W_O)
    att.W_O.data.add_(1.0)
    PACKS.clear()
    assert torch.equal(_unpacked(packed()), att.W_O)
    with torch.inference_mode():
        PACKS.clear()
        kept = packed()
    qkv = att._packed("qkv", torch.bfloat16, att.W_q, att.W_k, att.W_v)
    att.W_O.data.add_(1.0)
    att.W_k.data.add_(1.0)
    assert PACKS.refresh() >= 2
    assert packed() is kept and torch.equal(_unpacked(kept), att.W_O)
    assert torch.equal(_unpacked(qkv),
                       torch.cat((att.W_q, att.W_k, att.W_v), dim=1).to(torch.bfloat16))


def test_projection_packs_stay_with_their_module():
    """A deep copy or a pickled module starts with no packs and then keeps its own; a module
    that kept them in a dict before works on."""
    import copy
    import pickle

    from nanospeaker_amd.moe_kernel import PACKS

    att = _small_attention()
    att._packed("o", torch.float32, att.W_O)
    for other in (copy.deepcopy(att), pickle.loads(pickle.dumps(att))):
        assert len(other._packs) == 0 and len(att._packs) == 1
        with torch.no_grad():
            other.W_O.neg_()
        assert torch.equal(_unpacked(other._packed("o", torch.float32, other.W_O)), other.W_O)
        assert other._packs in PACKS._children
        PACKS.clear()
        assert len(other._packs) == 0
        att._packed("o", torch.float32, att.W_O)
    att._packs = {"o": ((), att.W_O.detach())}
    assert torch.equal(_unpacked(att._packed("o", torch.float32, att.W_O)), att.W_O)
