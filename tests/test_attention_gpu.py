"""The attention kernel (attention.hip) against softmax(scale Q K^T) V in 64 bits: tiles of 128 queries and 64 keys with every kind of
remainder, batches whose sequences start at any token, scores that make the running maximum move, one dominating key; and the
attention module of a model that uses it against the stock one."""
import pytest
import torch

from venom_amd import _lib, bert, spatha

pytestmark = pytest.mark.gpu


def exact(qkv, batch, seq, heads, scale):
    q, k, v = (t.double().reshape(batch, seq, heads, 64).transpose(1, 2).contiguous() for t in qkv.split(heads * 64, dim=1))
    scores = scale * (q.unsqueeze(3) * k.unsqueeze(2)).sum(-1) if seq <= 64 else scale * torch.matmul(q, k.transpose(2, 3).contiguous())
    return torch.matmul(torch.softmax(scores, -1), v).transpose(1, 2).reshape(batch, seq, heads * 64)


@pytest.mark.parametrize("batch,seq,heads", [(1, 1, 1), (2, 5, 16), (3, 31, 3), (1, 32, 16), (5, 33, 2), (2, 64, 4), (3, 65, 5), (2, 127, 16),
                                             (3, 127, 1), (2, 128, 3), (1, 129, 9), (2, 301, 4), (4, 512, 16), (1, 700, 2)])
@pytest.mark.parametrize("spread", [1.0, 8.0])
def test_attention_matches_the_exact_result(gpu, batch, seq, heads, spread):
    """Error bound: the probabilities and the result are rounded to fp16 (2^-11 each; the probabilities' roundings average over the
    keys but for a dominating one), scores and sums are fp32 (a score of 600 at spread 8 is off by 600 * 64 * 2^-24 at most):
    entries within 2^-9 of the largest |V| that they average, the whole within 6e-4."""
    gen = torch.Generator(device=gpu).manual_seed(seq * 7 + heads)
    qkv = torch.randn((batch * seq, 3 * heads * 64), generator=gen, device=gpu).half()
    qkv[:, :heads * 64] *= spread
    got = spatha._extension().attention(qkv, batch, seq, heads, 0.125)
    assert got.shape == (batch, seq, heads * 64) and got.dtype == torch.float16
    want = exact(qkv, batch, seq, heads, 0.125)
    diff = got.double() - want
    assert diff.norm().item() <= 6e-4 * want.norm().item()
    assert diff.abs().max().item() <= 2.0 ** -9 * qkv[:, 2 * heads * 64:].abs().max().item()
    # the buffer behind the view: padding columns are zero
    flat = torch.as_strided(got, (heads * 64, (batch * seq + 7) // 8 * 8), ((batch * seq + 7) // 8 * 8, 1))
    assert not flat[:, batch * seq:].any()


def test_attention_error_is_no_larger_than_the_stock_kernels(gpu):
    gen = torch.Generator(device=gpu).manual_seed(3)
    for batch, seq in ((2, 512), (2, 77)):
        qkv = torch.randn((batch * seq, 3072), generator=gen, device=gpu).half()
        want = exact(qkv, batch, seq, 16, 0.125)
        got = spatha._extension().attention(qkv, batch, seq, 16, 0.125)
        q, k, v = (t.reshape(batch, seq, 16, 64).transpose(1, 2) for t in qkv.split(1024, dim=1))
        stock = torch.nn.functional.scaled_dot_product_attention(q, k, v, scale=0.125).transpose(1, 2).reshape(batch, seq, 1024)
        ours, theirs = ((x.double() - want).norm().item() / want.norm().item() for x in (got, stock))
        print("relative error %.3g, the stock kernel's %.3g" % (ours, theirs))
        assert ours <= 1.02 * theirs          # (2 %: which way the roundings fall)


def test_attention_refuses_what_it_does_not_take(gpu):
    x = torch.zeros((8, 3 * 64), dtype=torch.float16, device=gpu)
    out = torch.zeros((64, 8), dtype=torch.float16, device=gpu)

    def call(head_dim=64, scale=0.125, pitch=192, out_pitch=8, q=x.data_ptr()):
        return _lib.lib().spatha_attention_f16(q, x.data_ptr(), x.data_ptr(), pitch, 1, 8, 1, head_dim, scale, out.data_ptr(), out_pitch,
                                               torch.cuda.current_stream().cuda_stream)
    assert call() == 0
    assert call(head_dim=32) == 3
    assert all(s != 0 for s in (call(scale=0.0), call(pitch=190), call(pitch=56), call(out_pitch=7), call(q=x.data_ptr() + 2), call(q=None)))
    assert spatha._extension().attention(x.float(), 1, 8, 1, 0.125) is None
    assert spatha._extension().attention(x, 2, 8, 1, 0.125) is None


@torch.no_grad()
def test_a_models_attention_takes_the_kernel_and_falls_back(gpu):
    """Without a mask the merged attention runs in the kernel; with one, in training mode or with a hook on a projection the stock
    forward answers.  Two fp16 attentions: 2e-3 apart at most (each within 6e-4 of the exact result)."""
    model = bert.merge_qkv(bert.linear_to_spmm(bert.build_bert_large(layers=1).to(gpu).half(), 2, 8, 64))
    stock = model.encoder.layer[0].attention.self
    x = torch.randn((2, 40, 1024), device=gpu).half()
    want, _ = stock(x)
    keys = list(model.state_dict())
    bert.fuse_add_layernorm(model, feature_major=True)
    att = model.encoder.layer[0].attention.self
    assert type(att) is bert.FusedSelfAttention and list(att.state_dict()) == [k[len("encoder.layer.0.attention.self."):] for k in keys
                                                                             if k.startswith("encoder.layer.0.attention.self.")]
    got, weights = att(x)
    assert weights is None and got.shape == want.shape and got.stride(-1) == 80
    assert (got.double() - want.double()).norm() <= 2e-3 * want.double().norm()
    mask = torch.ones((2, 1, 40, 40), dtype=torch.bool, device=gpu)
    mask[:, :, :, 30:] = False
    masked, _ = att(x, attention_mask=mask)
    assert masked.stride(-1) == 1 and not torch.equal(masked, got)
    handle = att.key.register_forward_hook(lambda m, a, o: o * 0)
    hooked, _ = att(x)
    handle.remove()
    v = att.value(x).float().mean(1, keepdim=True)
    assert (hooked.float() - v).abs().max() <= 4e-3       # equal scores: every token averages V
    assert torch.equal(att(x)[0], got)


def softmax_average(qkv, batch, seq, heads, scale):
    """`exact` with every product spelled out: an infinity or NaN meets the operands of its own query, key and feature only, and a
    probability of exactly zero takes no part."""
    q, k, v = (t.double().cpu().reshape(batch, seq, heads, 64).transpose(1, 2) for t in qkv.split(heads * 64, dim=1))
    p = torch.softmax(scale * (q.unsqueeze(3) * k.unsqueeze(2)).sum(-1), -1).unsqueeze(-1)          # [batch, heads, query, key, 1]
    terms = torch.where(p == 0, torch.zeros((), dtype=torch.float64), p * v.unsqueeze(2))
    return terms.sum(3).transpose(1, 2).reshape(batch, seq, heads * 64)


def same_kinds(got, want):
    """The same infinities and NaN in the same places, and the finite entries as near as in the tests above."""
    got, finite = got.double().cpu(), torch.isfinite(want)
    assert torch.equal(torch.isnan(got), torch.isnan(want))
    assert torch.equal(got[~finite & ~torch.isnan(want)], want[~finite & ~torch.isnan(want)])
    assert (got - want)[finite].norm() <= 6e-4 * want[finite].norm()


@pytest.mark.parametrize("seq", [1, 5, 40, 64, 65, 127, 130])
@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan")])
def test_an_infinity_in_the_last_value_reaches_its_feature_alone(gpu, seq, value):
    """Keys behind a sequence's end have probability zero, and zero times infinity would be NaN: their values have to be zeros."""
    gen = torch.Generator(device=gpu).manual_seed(seq)
    qkv = torch.randn((2 * seq, 3 * 2 * 64), generator=gen, device=gpu).half()
    qkv[seq - 1, 2 * 128 + 64 + 5] = value          # first sequence, second head, feature 5 of V
    got = spatha._extension().attention(qkv, 2, seq, 2, 0.125)
    same_kinds(got, softmax_average(qkv, 2, seq, 2, 0.125))


@pytest.mark.parametrize("seq,barred", [(65, 64), (130, 64), (130, 128), (200, 70), (96, 95)])
def test_keys_of_score_minus_infinity_take_no_part(gpu, seq, barred):
    """Whole tiles of them ahead of the first finite score leave nothing behind; a query with nothing else is NaN, as in torch's softmax."""
    gen = torch.Generator(device=gpu).manual_seed(seq + barred)
    qkv = torch.randn((2 * seq, 3 * 64), generator=gen, device=gpu).half()
    qkv[:, 3] = qkv[:, 3].abs() + 0.5             # feature 3 of every query is positive
    qkv[:barred, 64 + 3] = float("-inf")          # the first sequence's first keys
    qkv[seq:, 64 + 3] = float("-inf")             # every key of the second one
    got = spatha._extension().attention(qkv, 2, seq, 1, 0.125)
    want = softmax_average(qkv, 2, seq, 1, 0.125)
    assert torch.isfinite(want[0]).all() and torch.isnan(want[1]).all()
    same_kinds(got, want)


def fused_attention(gpu, layers=1):
    model = bert.merge_qkv(bert.linear_to_spmm(bert.build_bert_large(layers=layers).to(gpu).half(), 2, 8, 64))
    return bert.fuse_add_layernorm(model, feature_major=True).encoder.layer[0].attention.self


@torch.no_grad()
def test_the_fused_attention_keeps_no_product(gpu, monkeypatch):
    """Its projections have one reader: every forward computes them, and none outlives it (the three separate projections share theirs)."""
    att = fused_attention(gpu)
    group, x = att.query._group, torch.randn((2, 40, 1024), device=gpu).half()
    computed = []
    run = bert.SrnmSpmm._run_native
    monkeypatch.setattr(bert.SrnmSpmm, "_run_native", staticmethod(lambda *a, **k: computed.append(1) or run(*a, **k)))
    first = att(x)[0]
    assert len(computed) == 1 and group._last == (None, None, None)
    assert torch.equal(att(x)[0], first) and len(computed) == 2 and group._last == (None, None, None)
    q, k, v = att.query(x), att.key(x), att.value(x)
    assert len(computed) == 3 and torch.equal(group._last[2], torch.cat([q, k, v], -1).reshape(80, 3072))


def replaced(att):
    linear = torch.nn.Linear(1024, 1024, device=att.key.values.device, dtype=torch.float16)
    att.query = linear


class Doubling(bert.SrnmSpmm):
    def forward(self, input):
        return 2 * super().forward(input)


def subclassed(att):
    att.value.__class__ = Doubling


def own_forward(att):
    forward = att.value.forward
    att.value.forward = lambda x: 3 * forward(x)


@pytest.mark.parametrize("change", [replaced, subclassed, own_forward])
@torch.no_grad()
def test_projections_that_do_more_than_the_product_run(gpu, change):
    from transformers.models.bert.modeling_bert import BertSelfAttention

    att, x = fused_attention(gpu), torch.randn((2, 24, 1024), device=gpu).half()
    plain = att(x)[0]
    change(att)
    got = att(x)[0]
    assert torch.equal(got, BertSelfAttention.forward(att, x)[0]) and not torch.allclose(got, plain, atol=1e-2)


@torch.no_grad()
def test_a_hook_on_every_module_sees_the_projections(gpu):
    att, x, seen = fused_attention(gpu), torch.randn((2, 24, 1024), device=gpu).half(), []
    handle = torch.nn.modules.module.register_module_forward_hook(lambda m, a, o: seen.append(m))
    try:
        att(x)
    finally:
        handle.remove()
    assert all(any(m is p for m in seen) for p in (att.query, att.key, att.value))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@torch.no_grad()
def test_autocast_decides_the_type_of_the_context(gpu, dtype):
    from transformers.models.bert.modeling_bert import BertSelfAttention

    att, x = fused_attention(gpu), torch.randn((2, 24, 1024), device=gpu).half()
    with torch.autocast("cuda", dtype=dtype):
        got, want = att(x)[0], BertSelfAttention.forward(att, x)[0]
    assert got.dtype == want.dtype == dtype
    assert (got.double() - want.double()).norm() <= 2e-3 * want.double().norm()          # (two fp16 attentions, or the same bits)
