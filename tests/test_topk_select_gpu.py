"""Top-k selection of index scores on the GPU against the oracle, through the C ABI.
Integer work: the chosen indices and their order must be bit-exact."""
import pytest
import torch

from oracle import mla

pytestmark = pytest.mark.gpu


def run_kernel(capi, dev, scores, k, lengths=None):
    out = torch.full((scores.shape[0], k), -7, dtype=torch.int32, device=dev)
    capi.topk_select_launch(out, scores.to(dev), None if lengths is None else lengths.to(dev))
    torch.cuda.synchronize()
    return out.cpu()


@pytest.mark.parametrize('shape', [(3, 300, 40), (2, 32768, 2048), (5, 1000, 1000), (1, 5000, 1), (4, 70, 128),
                                   (2, 1024, 512), (3, 1025, 7), (2, 100000, 2048)])
def test_random_scores(capi, dev, shape):
    B, n, k = shape
    gen = torch.Generator().manual_seed(n + k)
    scores = torch.randn(B, n, generator=gen) * 3
    assert torch.equal(run_kernel(capi, dev, scores, k), mla.topk_select(scores, k))


def test_ties_specials_and_lengths(capi, dev):
    gen = torch.Generator().manual_seed(41)
    scores = torch.randint(-3, 4, (8, 3000), generator=gen).float()      # seven distinct values: ties everywhere
    scores[0, 5] = float('inf')
    scores[1, 7::11] = float('-inf')
    scores[2, 3::7] = float('nan')
    scores[3, ::2] = -0.0
    scores[3, 1::2] = 0.0
    scores[4] = 1.5                                                      # one value only
    scores[5] = float('nan')
    lengths = torch.tensor([3000, 2999, 1024, 1023, 1, 17, 0, 5000], dtype=torch.int32)
    for k in (1, 64, 1024, 2048, 3000, 3100):
        for ln in (None, lengths):
            got = run_kernel(capi, dev, scores, k, ln)
            assert torch.equal(got, mla.topk_select(scores, k, ln)), (k, ln is not None)


def test_denormals_and_close_values(capi, dev):
    # keys that differ only in the last byte, across zero
    base = torch.tensor([1e-42, -1e-42, 0.0, 1.0, 1.0 + 2 ** -23, 1.0 - 2 ** -24, -1.0, 3e38, -3e38])
    gen = torch.Generator().manual_seed(42)
    scores = base[torch.randint(0, base.numel(), (4, 4096), generator=gen)]
    for k in (1, 100, 2048, 4096):
        assert torch.equal(run_kernel(capi, dev, scores, k), mla.topk_select(scores, k))


def _rows(kind, n, gen):
    x = torch.randn(4, n, generator=gen)
    if kind == 'clustered':      # the large scores are neighbours: a sample of the row misjudges their number
        x[:, n // 3:n // 3 + 3000] += 6
    elif kind == 'distinct':     # few values: the threshold is shared by many entries
        x = (x * 8).round() / 8
    elif kind == 'wide':         # forty octaves, the threshold far above the sampled pivot or below zero
        x = torch.exp2(x * 10) * torch.where(torch.rand(4, n, generator=gen) < 0.01, 1.0, -1.0)
    elif kind == 'masked':       # fewer than k entries left above -inf
        x[torch.rand(4, n, generator=gen) < 0.95] = float('-inf')
        x[3] = torch.where(x[3] > 0, x[3], torch.full((), float('nan')))
    elif kind == 'two':          # two values, among them one pair that shares its upper digits
        x = (x > 0).float()
        x[2] += 1.0 / 1024 * x[2] + 1.0
        x[3] = x[3] * 2.0 ** -20 + 1.0
    elif kind == 'special':
        x[0, ::3] = float('nan')
        x[1, torch.rand(n, generator=gen) < 0.95] = float('-inf')
        x[2, ::2] = float('inf')
        x[3] = torch.where(x[3] > 1.5, x[3], torch.zeros(()))
    return x


@pytest.mark.parametrize('n', [600, 2500, 4096, 4097, 8192, 8193, 16385, 32768, 32769, 65536, 65537, 98305, 262144, 262145])
@pytest.mark.parametrize('kind', ['normal', 'clustered', 'distinct', 'wide', 'special', 'masked', 'two'])
def test_long_rows(capi, dev, n, kind):
    # edges of the row classes (in registers, read again, filtered or not), k at the limits of the candidate list
    gen = torch.Generator().manual_seed(n)
    scores = _rows(kind, n, gen)
    lengths = torch.tensor([n, n - 1, n // 2 + 7, 5000], dtype=torch.int32)
    for k, ln in ((2048, None), (2048, lengths), (1, None), (3072, lengths), (3073, None)):
        assert torch.equal(run_kernel(capi, dev, scores, k, ln), mla.topk_select(scores, k, ln)), (k, ln is not None)


@pytest.mark.parametrize('n', [16384, 32768, 65536])
@pytest.mark.parametrize('kind', ['normal', 'clustered', 'special', 'two'])
def test_lengths_around_the_words_of_a_wavefront(capi, dev, n, kind):
    # a row in registers is dealt out in 8 words of 64 entries per wavefront and step: one entry less and more than whole
    # steps, than what a wavefront takes of them, and than a word
    gen = torch.Generator().manual_seed(n)
    lengths = sorted({v for step in (8192, 16384, 24576, 40960, 57344, 65536) for v in (step - 1, step, step + 1)
                      if v <= n} | {1, 63, 64, 65, 511, 512, 513, 3000, 8192 + 512, 8192 + 513, 8192 + 1025})
    scores = _rows(kind, n, gen).repeat(-(-len(lengths) // 4), 1)[:len(lengths)]
    ln = torch.tensor(lengths, dtype=torch.int32)
    for k in (64, 2048):
        assert torch.equal(run_kernel(capi, dev, scores, k, ln), mla.topk_select(scores, k, ln)), k


def test_selected_indices_feed_the_attention(capi, dev):
    # selection -> sparse-MLA decode; shorter requests leave -1 entries, which the attention skips
    gen = torch.Generator().manual_seed(43)
    B, H, N, k = 3, 128, 1024, 256
    q, kv, _ = mla.mla_make_inputs(B, H, N, k, generator=gen)
    scores = torch.randn(B, N, generator=gen)
    lengths = torch.tensor([1024, 100, 300], dtype=torch.int32)
    idx = torch.empty(B, k, dtype=torch.int32, device=dev)
    capi.topk_select_launch(idx, scores.to(dev), lengths.to(dev))
    out = torch.empty(B, H, 512, dtype=torch.float32, device=dev)
    ws = torch.empty(capi.sparse_mla_workspace_bytes(B, H, k), dtype=torch.uint8, device=dev)
    capi.sparse_mla_decode_launch(out, q.to(dev), kv.to(dev), idx, ws)
    torch.cuda.synchronize()
    want_idx = mla.topk_select(scores, k, lengths)
    assert torch.equal(idx.cpu(), want_idx) and (want_idx[1] == -1).sum() == k - 100
    ref = mla.sparse_mla_decode(q, kv, want_idx, out_dtype=torch.float32)
    assert mla.rel_rms_error(out.cpu(), ref) <= 2e-2


def test_rejects_bad_arguments(capi, dev):
    with pytest.raises(ValueError):
        capi.topk_select_launch(torch.zeros(2, 4, dtype=torch.int32, device=dev),
                                torch.zeros(2, 8, dtype=torch.float64, device=dev))
