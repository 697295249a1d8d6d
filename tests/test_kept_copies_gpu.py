"""What a layer keeps of one call for the next (the transposed copy of an activation, the merged projections' result) belongs to
the stream and the graph capture that it was computed on."""
import pytest
import torch

from venom_amd import bert, spatha
from venom_amd.bert import SrnmSpmm

pytestmark = pytest.mark.gpu

TOKENS = [8, 24, 301]          # read as they lie; through a kept copy; through a kept copy with padded rows


def _layer(gpu, seed=0, rows=64):
    torch.manual_seed(seed)
    return SrnmSpmm(torch.nn.Linear(128, rows).half().to(gpu), 2, 8, 64, magnitude=True)


def _direct(layer, x):
    return spatha.spmm(layer.metadata, layer.columns, layer.values, x.T.contiguous(), layer.bias, layer.nrows_sp, layer.ncols_sp,
                       x.shape[0], layer.v, layer.n, layer.m)


def _merged(gpu):
    layers = [_layer(gpu, seed, 64) for seed in range(3)]
    return layers, bert._MergedProjections(layers)


def test_a_kept_copy_is_not_taken_on_another_stream(gpu):
    layer, x = _layer(gpu), torch.randn(24, 128, device=gpu).half()
    want = _direct(layer, x)
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream(device=gpu) for _ in range(2)]
    kept = []
    with torch.no_grad():
        for s in streams:
            with torch.cuda.stream(s):
                for _ in range(2):
                    assert torch.equal(layer(x), want)
                    kept.append(SrnmSpmm._last_rhs[2])
            s.synchronize()
    assert kept[0] is kept[1] and kept[2] is kept[3]            # shared on one stream
    assert kept[1].data_ptr() != kept[2].data_ptr()             # made anew on the other


def test_the_general_path_keeps_by_stream_too(gpu):
    x, x_t = torch.randn(24, 128, device=gpu).half(), torch.randn(128, 24, device=gpu).half()
    torch.cuda.synchronize()
    SrnmSpmm.offer_transposed(x, x_t)
    assert SrnmSpmm._transposed(x) is x_t or SrnmSpmm._transposed(x).data_ptr() == x_t.data_ptr()
    s = torch.cuda.Stream(device=gpu)
    with torch.cuda.stream(s):
        copy = SrnmSpmm._transposed(x)
        assert copy.data_ptr() != x_t.data_ptr() and torch.equal(copy, x.T)
    s.synchronize()


def test_merged_projections_keep_by_stream(gpu):
    layers, group = _merged(gpu)
    x = torch.randn(24, 128, device=gpu).half()
    torch.cuda.synchronize()
    with torch.no_grad():
        group.output(0, 64, x)
        first = group._last[2]
        assert torch.equal(group.output(1, 64, x), _direct(layers[1], x)) and group._last[2] is first
        s = torch.cuda.Stream(device=gpu)
        with torch.cuda.stream(s):
            assert torch.equal(group.output(1, 64, x), _direct(layers[1], x))
            assert group._last[2] is not first
        s.synchronize()


@pytest.mark.parametrize("tokens", TOKENS)
@pytest.mark.parametrize("kind", ["layer", "merged"])
def test_a_graph_replays_on_new_contents_of_an_input_it_was_warmed_up_on(gpu, tokens, kind):
    """The usual order: a warm-up on the input, a capture on the same stream, replays on new contents; the eager call after them."""
    if kind == "layer":
        layer = _layer(gpu)
        call, want = layer, lambda x: _direct(layer, x)
    else:
        layers, group = _merged(gpu)
        call = lambda x: torch.stack([group.output(i, 64, x) for i in range(3)])
        want = lambda x: torch.stack([_direct(l, x) for l in layers])
    x = torch.randn(tokens, 128, device=gpu).half()
    s = torch.cuda.Stream(device=gpu)
    s.wait_stream(torch.cuda.current_stream(gpu))
    graphs, results = [], []
    with torch.no_grad(), torch.cuda.stream(s):
        call(x)
        for _ in range(2):                  # the second graph must not read what only the first one's replay writes
            graphs.append(torch.cuda.CUDAGraph())
            with torch.cuda.graph(graphs[-1], stream=s):
                results.append(call(x))
        eager = call(x)                     # nothing that was recorded has run yet
        assert torch.equal(eager, want(x))
        for seed in range(3):
            x.copy_(torch.randn(tokens, 128, device=gpu).half())
            for i in (1, 0):
                graphs[i].replay()
                s.synchronize()
                assert torch.equal(results[i], want(x)), (seed, i)
            assert torch.equal(call(x), want(x))
    s.synchronize()
