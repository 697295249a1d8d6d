"""The embedding kernel (three table rows, two additions, LayerNorm; layernorm.hip) against the stock module's own operations, and the
norm that pads its feature-major copy for any token count."""
import ctypes

import pytest
import torch

from venom_amd import _lib, bert, spatha

pytestmark = pytest.mark.gpu


def close(got, want):
    """Statistics in another order: neighbouring fp16 values at most, nearly all equal (as for add_layernorm)."""
    diff = (got.float() - want.float()).abs()
    return (got == want).float().mean().item() >= 0.99 and bool((diff <= torch.maximum(want.float().abs() * 2.0 ** -10, torch.tensor(1e-3).to(diff))).all())


@pytest.mark.parametrize("batch,seq", [(1, 1), (2, 5), (3, 31), (1, 33), (2, 324), (5, 77), (4, 512)])
@pytest.mark.parametrize("types", [None, "given"])
@torch.no_grad()
def test_fused_embedding_equals_the_stock_module(gpu, batch, seq, types):
    stock = bert.build_bert_large(layers=1).to(gpu).half()
    fused = bert.fuse_add_layernorm(bert.merge_qkv(bert.linear_to_spmm(bert.build_bert_large(layers=1).to(gpu).half(), 2, 8, 64)), feature_major=True)
    emb = fused.embeddings
    assert type(emb) is bert.FusedEmbeddings and list(emb.state_dict()) == list(stock.embeddings.state_dict())
    ids = torch.randint(0, 30522, (batch, seq), device=gpu)
    tt = None if types is None else torch.randint(0, 2, (batch, seq), device=gpu)
    want = stock.embeddings(input_ids=ids, token_type_ids=tt)
    got = emb(input_ids=ids, token_type_ids=tt)
    assert got.shape == want.shape and got.is_contiguous() and close(got, want)
    # the copy that it hands on: padded rows, zeros behind the last token
    copy, tokens = bert.SrnmSpmm._last_rhs[2], batch * seq
    assert tuple(copy.shape) == (1024, tokens) and torch.equal(copy.t(), got.reshape(tokens, 1024))
    padded = torch.as_strided(copy, (1024, copy.stride(0)), copy.stride())
    assert copy.stride(0) == (tokens + 7) // 8 * 8 and not padded[:, tokens:].any()
    # calls that the kernel does not take answer as the stock module does
    position = torch.arange(seq, device=gpu).flip(0)[None]
    assert torch.equal(emb(input_ids=ids, position_ids=position), stock.embeddings(input_ids=ids, position_ids=position))
    x = torch.randn((batch, seq, 1024), device=gpu).half()
    assert torch.equal(emb(inputs_embeds=x), stock.embeddings(inputs_embeds=x))
    with torch.enable_grad():
        assert emb(input_ids=ids).requires_grad


@pytest.mark.parametrize("tokens,hidden", [(1, 1024), (7, 512), (33, 1024), (75, 768), (1037, 1280), (9, 4096), (130, 72)])
def test_padded_feature_major_norm(gpu, tokens, hidden):
    gen = torch.Generator(device=gpu).manual_seed(tokens + hidden)
    x, r = (torch.randn((tokens, hidden), generator=gen, device=gpu).half() for _ in range(2))
    w, b = ((0.1 * torch.randn(hidden, generator=gen, device=gpu)).half() for _ in range(2))
    want = spatha.add_layernorm(x, r, w, b, 1e-12)
    out, copy = spatha._extension().add_layernorm(x, r, w, b, 1e-12, True)
    pitch = (tokens + 7) // 8 * 8
    assert torch.equal(out, want) and torch.equal(copy, want.t()) and copy.stride() == (pitch, 1)
    guard = torch.full((hidden * pitch + 128,), 7.0, dtype=torch.float16, device=gpu)
    stream = ctypes.c_void_p(torch.cuda.current_stream(gpu).cuda_stream)
    _lib.check(_lib.lib().spatha_add_layernorm_f16_tp(x.data_ptr(), r.data_ptr(), w.data_ptr(), b.data_ptr(), 1e-12, tokens, hidden,
                                                      out.data_ptr(), guard[64:].data_ptr(), stream), "ln_tp")
    padded = guard[64:-64].view(hidden, pitch)
    assert torch.equal(padded[:, :tokens], want.t()) and not padded[:, tokens:].any()
    assert bool((guard[:64] == 7.0).all()) and bool((guard[-64:] == 7.0).all())


def one_embedding(gpu):
    return bert.fuse_add_layernorm(bert.build_bert_large(layers=1).to(gpu).half()).embeddings


@torch.no_grad()
def test_autocast_decides_the_type_of_the_embedding(gpu):
    """Under autocast LayerNorm runs, and answers, in fp32."""
    from transformers.models.bert.modeling_bert import BertEmbeddings

    emb, ids = one_embedding(gpu), torch.randint(0, 30522, (2, 24), device=gpu)
    with torch.autocast("cuda", dtype=torch.float16):
        got, want = emb(input_ids=ids), BertEmbeddings.forward(emb, ids)
    assert want.dtype == torch.float32 and got.dtype == torch.float32 and torch.equal(got, want)


@torch.no_grad()
def test_a_trace_of_the_embedding_follows_its_ids(gpu):
    from transformers.models.bert.modeling_bert import BertEmbeddings

    emb = one_embedding(gpu)
    first, second = (torch.randint(0, 30522, (2, 24), device=gpu) for _ in range(2))
    traced = torch.jit.trace(emb, (first,), check_trace=False)
    assert torch.equal(traced(second), BertEmbeddings.forward(emb, second))


@torch.no_grad()
def test_transformed_weights_take_the_stock_embedding(gpu):
    """Tables in batches (vmap) and tables with tangents (forward-mode differentiation)."""
    emb, ids = one_embedding(gpu), torch.randint(0, 30522, (2, 24), device=gpu)
    table = emb.word_embeddings.weight
    tables = torch.stack([table, 2 * table])
    call = lambda w: torch.func.functional_call(emb, {"word_embeddings.weight": w}, (ids,))
    got = torch.vmap(call)(tables)
    assert got.shape == (2, 2, 24, 1024) and all(close(g, call(w)) for g, w in zip(got, tables))
    _, tangent = torch.func.jvp(call, (table,), (table,))
    assert float(tangent.abs().max()) > 0


@pytest.mark.parametrize("feature_major", [False, True])
@pytest.mark.parametrize("batch,seq", [(1, 1), (2, 31), (3, 512)])
@torch.no_grad()
def test_the_models_own_types_go_by_position(gpu, feature_major, batch, seq):
    """The stock module looks its row of token types up at the position ids, and takes a caller's as they lie."""
    from transformers.models.bert.modeling_bert import BertEmbeddings

    emb = one_embedding(gpu)
    emb.feature_major = feature_major
    emb.token_type_ids = (torch.arange(512, device=gpu) * 7 // 5 % 2)[None]
    emb.position_ids = (torch.arange(512, device=gpu) * 5 + 3).remainder(512)[None]
    ids = torch.randint(0, 30522, (batch, seq), device=gpu)
    for types in (None, emb.token_type_ids[:, :seq], emb.token_type_ids[:, :seq].expand(batch, seq).contiguous()):
        assert close(emb(input_ids=ids, token_type_ids=types), BertEmbeddings.forward(emb, ids, types))


@pytest.mark.parametrize("tokens", [7, 8])
def test_norms_run_in_inference_mode(gpu, tokens):
    """Its tensors have no version to know a handed-on copy by: none is offered."""
    norm = bert.fuse_add_layernorm(bert.build_bert_large(layers=1).to(gpu).half(), feature_major=True).encoder.layer[0].attention.output
    x, r = (torch.randn((1, tokens, 1024), device=gpu).half() for _ in range(2))
    with torch.no_grad():
        want = norm(x, r)
    with torch.inference_mode():
        assert torch.equal(norm(x, r), want)


@pytest.mark.parametrize("batch,seq", [(3, 37), (2, 64)])
@torch.no_grad()
def test_the_whole_fused_encoder_tracks_the_unfused_one(gpu, monkeypatch, batch, seq):
    """Every fusion at once, two layers: the kernels run, every right-hand side is handed on (no layer makes a transposed copy of its own),
    and the last hidden state is the unfused layers'.  Each is off by 7e-4 (norm) from the same encoder in fp32: twice that apart."""
    def build():
        torch.manual_seed(11)
        return bert.linear_to_spmm(bert.build_bert_large(layers=2).to(gpu).half(), 2, 8, 64, magnitude=True)

    plain = build()
    fused = bert.fuse_add_layernorm(bert.merge_qkv(bert.fuse_feed_forward(build(), activation_in_kernel=True)), feature_major=True)
    ext, calls, copies = spatha._extension(), [], []

    def counted(name):
        native = getattr(ext, name)

        def call(*args):
            calls.append(name)
            got = native(*args)
            assert got is not None
            if name == "layer_spmm" and got[1] is not None:
                copies.append(args[0].shape)
            return got
        monkeypatch.setattr(ext, name, call)

    ids = torch.randint(0, 30522, (batch, seq), device=gpu)
    want = plain(ids).last_hidden_state
    for name in ("embed_layernorm", "layer_spmm", "attention", "add_layernorm"):
        counted(name)
    got = fused(ids).last_hidden_state
    one = ["layer_spmm", "attention", "layer_spmm", "add_layernorm", "layer_spmm", "layer_spmm", "add_layernorm"]
    assert calls == ["embed_layernorm"] + 2 * one and not copies
    assert (got.double() - want.double()).norm() <= 1.4e-3 * want.double().norm()
