"""Which calls the fused embedding and attention modules take, and which they leave to the stock modules: hooks, replaced and
subclassed parts, operands of other shapes and places.  Runs on the CPU with a stand-in for the library's kernels; what the kernels
compute is in test_embedding_gpu.py and test_attention_gpu.py."""
import types

import pytest
import torch

from venom_amd import bert, spatha

TAKEN = 7.0          # what the stand-in answers


@pytest.fixture
def kernels(monkeypatch):
    """The calls that reach the library."""
    calls = []

    def embed_layernorm(ids, *args):
        calls.append(args)
        return torch.full((*ids.shape, 64), TAKEN), None

    have = {"embed_layernorm": embed_layernorm}
    monkeypatch.setattr(spatha, "_extension", lambda: types.SimpleNamespace(**have))
    monkeypatch.setattr(spatha, "_native", have.get)
    return calls


def make_embeddings():
    from transformers.models.bert.modeling_bert import BertConfig, BertEmbeddings

    torch.manual_seed(0)
    return BertEmbeddings(BertConfig(hidden_size=64, num_hidden_layers=1, num_attention_heads=1, intermediate_size=64, vocab_size=50)).eval()


def fused_embeddings():
    holder = torch.nn.ModuleDict({"embeddings": make_embeddings()})
    return bert.fuse_add_layernorm(holder)["embeddings"]


class DoubledNorm(torch.nn.LayerNorm):
    def forward(self, x):
        return 2 * super().forward(x)


class ScaledNorm(torch.nn.Module):
    """Another norm with a LayerNorm's attributes."""

    def __init__(self, like):
        super().__init__()
        self.weight, self.bias, self.eps = like.weight, like.bias, like.eps

    def forward(self, x):
        return x * self.weight


def doubled(module, args, out):
    return 2 * out


def change_nothing(e):
    pass


def own_forward(e):
    e.LayerNorm.forward = lambda x: 3 * x


def subclassed(e):
    norm = DoubledNorm(64)
    norm.load_state_dict(e.LayerNorm.state_dict())
    e.LayerNorm = norm


def live_dropout(e):
    torch.manual_seed(5)
    e.dropout.train()


CHANGES = [lambda e: e.LayerNorm.register_forward_hook(doubled), lambda e: e.LayerNorm.register_forward_pre_hook(lambda m, a: (2 * a[0] + 1,)),
           lambda e: e.dropout.register_forward_hook(doubled), lambda e: e.dropout.register_forward_pre_hook(lambda m, a: (2 * a[0],)),
           lambda e: e.word_embeddings.register_forward_hook(doubled), own_forward, subclassed,
           lambda e: setattr(e, "LayerNorm", ScaledNorm(e.LayerNorm)), lambda e: setattr(e, "dropout", torch.nn.Tanh()), live_dropout]


@pytest.mark.parametrize("change", [change_nothing] + CHANGES)
def test_embedding_parts_that_do_more_than_the_kernel_run(kernels, change):
    stock, fused = make_embeddings(), fused_embeddings()
    ids = torch.arange(12).reshape(2, 6)
    with torch.no_grad():
        change(stock)
        want = stock(input_ids=ids)
        change(fused)
        got = fused(input_ids=ids)
    if change is change_nothing:
        assert len(kernels) == 1 and bool((got == TAKEN).all())
    else:
        assert not kernels and torch.equal(got, want)


def test_a_hook_on_every_module_sees_the_embeddings_norm(kernels):
    fused, seen = fused_embeddings(), []
    handle = torch.nn.modules.module.register_module_forward_hook(lambda m, a, o: seen.append(type(m)))
    try:
        with torch.no_grad():
            fused(input_ids=torch.arange(6)[None])
    finally:
        handle.remove()
    assert not kernels and torch.nn.LayerNorm in seen


@pytest.mark.parametrize("batch,seq,types,taken", [(2, 6, (2, 6), True), (2, 6, (1, 6), True), (1, 6, (1, 6), True), (2, 6, None, True),
                                                   (2, 6, (1, 9), False), (1, 6, (1, 512), False), (1, 1, (1, 9), False), (2, 1, (1, 2), False),
                                                   (2, 6, (1, 1), False), (2, 6, (2, 1), False)])
def test_token_types_of_a_caller_have_the_ids_length(kernels, batch, seq, types, taken):
    """The model's own row of token types is longer than the sequence; a caller's is not."""
    stock, fused = make_embeddings(), fused_embeddings()
    ids = torch.arange(batch * seq).reshape(batch, seq)
    tt = None if types is None else torch.ones(types, dtype=torch.int64)

    def answer(module):
        with torch.no_grad():
            try:
                return module(input_ids=ids, token_type_ids=tt)
            except RuntimeError:
                return "refused"

    want, got = answer(stock), answer(fused)
    assert bool(kernels) == taken
    if not taken:
        assert got == want if isinstance(want, str) else torch.equal(got, want)


def test_the_embedding_needs_no_extension(monkeypatch):
    """A dense model, on the CPU here, asks for none: the stock forward answers where there is no extension and where there is one."""
    import sys

    import venom_amd

    ids = torch.arange(12).reshape(2, 6)
    with torch.no_grad():
        want = make_embeddings()(input_ids=ids)
        assert torch.equal(fused_embeddings()(input_ids=ids), want)
        monkeypatch.setitem(sys.modules, "venom_amd._spatha_torch", None)       # importing it raises ImportError
        monkeypatch.delattr(venom_amd, "_spatha_torch", raising=False)
        monkeypatch.setattr(spatha, "_loaded_extension", None)
        monkeypatch.setattr(spatha, "_extension_absent", False)
        assert torch.equal(fused_embeddings()(input_ids=ids), want)


def test_the_embedding_goes_with_the_default_build_only(monkeypatch):
    """Where SPATHA_LIBRARY names another build, the extension, which is linked to the default one, is not asked."""
    from venom_amd import _lib

    monkeypatch.setattr(_lib, "IS_DEFAULT_BUILD", False)
    monkeypatch.setattr(spatha, "_extension", lambda: pytest.fail("the extension was asked"))
    with torch.no_grad():
        fused_embeddings()(input_ids=torch.arange(6)[None])


def merged(cols, rows):
    """A _MergedProjections without matrices: its product is x times the number of the call."""

    class Merged(bert._MergedProjections):
        def __init__(self):
            self.starts, self.rows, self._last, self.calls = [0], rows, (None, None, None), 0

        def product(self, flat):
            self.calls += 1
            return flat[:, :rows] * self.calls

    return Merged


def test_a_product_of_another_thread_is_not_taken():
    """Between keeping a product and answering from it another thread may keep its own."""
    mine, others = torch.randn(6, 8), torch.randn(4, 8)

    class Raced(merged(8, 4)):
        def __setattr__(self, name, value):
            super().__setattr__(name, value)
            if name == "_last" and value[0] is not None:
                self.__dict__["_last"] = (bert._activation_key(others), others, others[:, :4])

    group = Raced()
    assert torch.equal(group.output(0, 4, mine), mine[:, :4])
    assert torch.equal(group.output(0, 4, mine), mine[:, :4] * 2)          # (what is kept is the other thread's: computed again)


def test_a_transposed_copy_of_another_thread_is_not_taken():
    mine, others = torch.randn(6, 8), torch.randn(4, 8)
    entries = [(bert._activation_key(mine), mine, mine.t().contiguous())]

    class Raced(type(bert.SrnmSpmm)):
        @property
        def _last_rhs(cls):
            seen = entries[-1]
            entries.append((bert._activation_key(others), others, others.t().contiguous()))         # between two looks
            return seen

        @_last_rhs.setter
        def _last_rhs(cls, value):
            entries.append(value)

    class Layer(bert.SrnmSpmm, metaclass=Raced):
        pass

    assert torch.equal(Layer._transposed(mine), mine.t())
