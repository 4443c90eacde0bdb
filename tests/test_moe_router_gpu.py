"""Group-limited, bias-corrected routing on the GPU against the oracle, through the C ABI.

Bar: expert ids bit-exact, in the oracle's order (descending choice value, ties to the lower id). The kernel's
sigmoid and the oracle's may round differently in the last place, so a token whose decision hangs on two choice
values (or two group values) a few ulp apart may differ; such tokens are counted and must stay below 1 in 1000
(none occurs at the seeds used here up to 1000 tokens). Weights: rtol 1e-5."""
from pathlib import Path

import numpy as np
import pytest
import torch

from oracle import moe

pytestmark = pytest.mark.gpu


def run_kernel(capi, dev, logits, bias, k, G, kg, norm=True, scale=1.0):
    T = logits.shape[0]
    ids = torch.full((T, k), -1, dtype=torch.int32, device=dev)
    w = torch.full((T, k), float('nan'), device=dev)
    capi.moe_route_grouped_launch(ids, w, logits.to(dev), None if bias is None else bias.to(dev), G, kg, norm, scale)
    torch.cuda.synchronize()
    return ids.cpu(), w.cpu()


def check(capi, dev, logits, bias, k, G, kg, norm=True, scale=1.0):
    want_ids, want_w, choice = moe.route_grouped(logits, bias, k, G, kg, norm, scale)
    ids, w = run_kernel(capi, dev, logits, bias, k, G, kg, norm, scale)
    same = (ids == want_ids).all(dim=1)
    close_calls = 0
    for t in torch.nonzero(~same).flatten().tolist():
        assert len(set(ids[t].tolist())) == k
        a, b = set(ids[t].tolist()), set(want_ids[t].tolist())
        if a == b:      # same experts in another order: two of them must tie within a few ulp
            vals = choice[t][ids[t].long()].sort().values
            assert (vals[1:] - vals[:-1]).min() <= 4 * 2.0 ** -23 * vals.abs().max().clamp_min(1.0)
        close_calls += 1
    assert close_calls <= max(1, logits.shape[0] // 1000), close_calls
    torch.testing.assert_close(w[same], want_w[same], rtol=1e-5, atol=1e-9)
    return ids, w


@pytest.mark.parametrize('shape', [(64, 256, 8, 8, 4), (1000, 256, 8, 8, 4), (37, 64, 6, 4, 2), (5, 32, 4, 1, 1),
                                   (130, 512, 8, 16, 5), (9, 8, 2, 8, 3), (64, 384, 8, 8, 4), (3, 24, 5, 3, 2),
                                   (50, 128, 8, 8, 4), (21, 65, 6, 5, 2), (40, 64, 8, 2, 1), (30, 60, 4, 30, 9)])   # 1 to 32 lanes a group
@pytest.mark.parametrize('norm,scale', [(True, 2.5), (False, 1.0)])
def test_matches_oracle(capi, dev, shape, norm, scale):
    T, E, k, G, kg = shape
    gen = torch.Generator().manual_seed(T + E)
    logits = torch.randn(T, E, generator=gen)
    bias = 0.2 * torch.randn(E, generator=gen)
    check(capi, dev, logits, bias, k, G, kg, norm, scale)
    check(capi, dev, logits, None, k, G, kg, norm, scale)


def test_prefill_size_and_biased_experts(capi, dev):
    gen = torch.Generator().manual_seed(77)
    logits = torch.randn(8192, 256, generator=gen)
    logits[:, torch.randperm(256, generator=gen)[:16]] += 2.0
    bias = 0.1 * torch.randn(256, generator=gen)
    ids, w = check(capi, dev, logits, bias, 8, 8, 4, True, 2.5)
    assert all(len(set(r.tolist())) <= 4 for r in (ids[:500] // 32))
    torch.testing.assert_close(w.sum(dim=1), torch.full((8192,), 2.5), rtol=1e-5, atol=0)


def test_one_group_without_bias_is_the_plain_router(capi, dev):
    gen = torch.Generator().manual_seed(78)
    logits = torch.randn(300, 256, generator=gen).to(dev)
    ids = torch.empty(300, 8, dtype=torch.int32, device=dev)
    w = torch.empty(300, 8, device=dev)
    capi.moe_route_launch(ids, w, logits)
    ids2, w2 = run_kernel(capi, dev, logits.cpu(), None, 8, 1, 1)
    torch.cuda.synchronize()
    assert torch.equal(ids.cpu(), ids2)
    torch.testing.assert_close(w.cpu(), w2, rtol=1e-6, atol=0)


def test_ties_go_to_the_lower_group_and_the_lower_expert(capi, dev):
    logits = torch.zeros(4, 64)
    ids, w = run_kernel(capi, dev, logits, None, 6, 8, 2)
    assert torch.equal(ids, torch.tensor([[0, 1, 2, 3, 4, 5]] * 4, dtype=torch.int32))
    torch.testing.assert_close(w, torch.full((4, 6), 1 / 6), rtol=1e-6, atol=0)
    logits[:, 40:48] = 1.0          # group 5 now wins, group 0 is second
    ids, _ = run_kernel(capi, dev, logits, None, 6, 8, 2)
    assert torch.equal(ids, torch.tensor([[40, 41, 42, 43, 44, 45]] * 4, dtype=torch.int32))
    ids, _ = run_kernel(capi, dev, logits, None, 10, 8, 2)
    assert torch.equal(ids[0], torch.tensor([40, 41, 42, 43, 44, 45, 46, 47, 0, 1], dtype=torch.int32))


@pytest.mark.parametrize('E,G', [(64, 8), (128, 8), (96, 8), (192, 8), (256, 8), (320, 5), (384, 8), (512, 16), (60, 30)])
def test_rows_off_16_bytes_and_ties(capi, dev, E, G):
    # 1 to 8 experts a lane, groups in registers and not; rows that start off 16 bytes, equal values in one lane and in several
    gen = torch.Generator().manual_seed(E)
    logits = torch.randint(-3, 4, (33, E), generator=gen).float()
    store = torch.empty(33 * E + 1, device=dev)
    off = store[1:].view(33, E).copy_(logits)
    want_ids, _, _ = moe.route_grouped(logits, None, 4, G, 2)
    ids, w = torch.empty(33, 4, dtype=torch.int32, device=dev), torch.empty(33, 4, device=dev)
    capi.moe_route_grouped_launch(ids, w, off, None, G, 2)
    assert torch.equal(ids.cpu(), want_ids)
    want_ids, want_w = moe.route(logits, 4)
    capi.moe_route_launch(ids, w, off)
    assert torch.equal(ids.cpu(), want_ids)
    torch.testing.assert_close(w.cpu(), want_w, rtol=1e-6, atol=0)


def test_third_party_golden_fixture(capi, dev):
    z = np.load(Path(__file__).parent / 'golden' / 'router_golden.npz')
    for tag in 'abc':
        k, G, kg, norm = (int(v) for v in z[f'{tag}_params'])
        ids, w = run_kernel(capi, dev, torch.from_numpy(z[f'{tag}_logits']), torch.from_numpy(z[f'{tag}_bias']),
                            k, G, kg, bool(norm), float(z[f'{tag}_scale'][0]))
        order = ids.argsort(dim=-1)
        np.testing.assert_array_equal(ids.gather(1, order).numpy(), z[f'{tag}_ids'])
        np.testing.assert_allclose(w.gather(1, order).numpy(), z[f'{tag}_weights'], rtol=1e-5)


def test_rejects_unsupported_shapes(capi, dev):
    logits = torch.zeros(2, 256, device=dev)
    ids = torch.zeros(2, 8, dtype=torch.int32, device=dev)
    w = torch.zeros(2, 8, device=dev)
    for G, kg in ((7, 2), (8, 9), (128, 4), (8, 0)):
        with pytest.raises(capi.LaunchRejected):
            capi.moe_route_grouped_launch(ids, w, logits, None, G, kg)
    ids = torch.zeros(2, 40, dtype=torch.int32, device=dev)    # 40 experts wanted, 32 stay
    w = torch.zeros(2, 40, device=dev)
    with pytest.raises(capi.LaunchRejected):
        capi.moe_route_grouped_launch(ids, w, logits, None, 8, 1)
    torch.cuda.synchronize()


# ---- router projection ---------------------------------------------------------------------------

def run_logits(capi, dev, x, w):
    T, H = x.shape
    E = w.shape[0]
    logits = torch.full((T, E), float('nan'), device=dev)
    nbytes = capi.moe_router_logits_workspace_bytes(T, H, E)
    ws = torch.empty(nbytes, dtype=torch.uint8, device=dev) if nbytes else None
    capi.moe_router_logits_launch(logits, x.to(dev), w.to(dev), ws)
    torch.cuda.synchronize()
    return logits.cpu()


def logits_bound(x, w):
    # fp32 accumulation of H products in any order: |err| <= H * 2^-24 * sum |x_h w_eh| (loose by sqrt(H))
    return x.shape[1] * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)


@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float32])
@pytest.mark.parametrize('shape', [(64, 7168, 256), (1, 64, 32), (100, 448, 72), (700, 1024, 256), (33, 128, 1),
                                   (130, 2048, 384)])
def test_router_logits_match_float64(capi, dev, shape, dtype):
    T, H, E = shape
    gen = torch.Generator().manual_seed(T + E)
    x = torch.randn(T, H, generator=gen).to(dtype)
    w = torch.randn(E, H, generator=gen) * H ** -0.5
    got = run_logits(capi, dev, x, w)
    want = x.double() @ w.double().T
    assert torch.isfinite(got).all()
    assert ((got.double() - want).abs() <= logits_bound(x, w)).all()
    # as close to the exact product as the oracle's own fp32 evaluation
    err = (got.double() - want).abs().max().item()
    ref_err = (moe.router_logits(x, w).double() - want).abs().max().item()
    assert err <= 4 * ref_err + 1e-7


def test_router_logits_exact_on_integers(capi, dev):
    # small integers: every partial sum is an exact fp32 integer, so any summation order gives the same bits
    gen = torch.Generator().manual_seed(51)
    x = torch.randint(-8, 9, (96, 512), generator=gen).float().bfloat16()
    w = torch.randint(-8, 9, (64, 512), generator=gen).float()
    assert torch.equal(run_logits(capi, dev, x, w), x.float() @ w.T)


def test_router_logits_golden_fixture(capi, dev):
    z = np.load(Path(__file__).parent / 'golden' / 'router_golden.npz')
    for tag in 'a':                       # (the other two cases have hidden = 32, below the kernel's 64 grain)
        got = run_logits(capi, dev, torch.from_numpy(z[f'{tag}_hidden']).bfloat16(), torch.from_numpy(z[f'{tag}_weight']))
        torch.testing.assert_close(got, torch.from_numpy(z[f'{tag}_logits']), rtol=1e-5, atol=1e-6)


@pytest.mark.parametrize('shape', [(64, 8), (128, 8), (256, 8), (512, 8), (64, 32), (60, 3), (512, 64)])
def test_grouped_routing_passes_nan_over(capi, dev, shape):
    # a NaN score adds nothing to its group's value, wherever it stands beside the group's largest: every pair of
    # positions in group 0, which with the NaN left out is worth less than group 1 (two scores of 0.69 against one of 0.88)
    E, G = shape
    size = E // G
    at = torch.tensor([(i, j) for i in range(size) for j in range(size) if i != j])
    logits = torch.full((len(at), E), -6.0)
    logits[:, size:size + 2] = 0.8
    rows = torch.arange(len(at))
    logits[rows, at[:, 0]] = 2.0
    want_ids, want_w, _ = moe.route_grouped(logits, None, 2, G, 1)
    logits[rows, at[:, 1]] = float('nan')
    ids = torch.empty(len(at), 2, dtype=torch.int32, device=dev)
    w = torch.empty(len(at), 2, device=dev)
    capi.moe_route_grouped_launch(ids, w, logits.to(dev), None, G, 1)
    assert torch.equal(ids.cpu(), want_ids)
    torch.testing.assert_close(w.cpu(), want_w, rtol=1e-6, atol=1e-7)


def test_projection_then_grouped_routing_at_prefill_size(capi, dev):
    # hidden states -> logits -> experts, against the oracle's chain; a token may differ only on a near-tie
    gen = torch.Generator().manual_seed(52)
    T, H, E = 8192, 1024, 256
    x = torch.randn(T, H, generator=gen).bfloat16()
    w = torch.randn(E, H, generator=gen) * H ** -0.5
    bias = 0.1 * torch.randn(E, generator=gen)
    logits = run_logits(capi, dev, x, w)
    ids, _ = run_kernel(capi, dev, logits, bias, 8, 8, 4, True, 2.5)
    want_ids, _, _ = moe.route_grouped(moe.router_logits(x, w), bias, 8, 8, 4, True, 2.5)
    differing = (ids != want_ids).any(dim=1).sum().item()
    assert differing <= 8, differing        # logits differ in the last place: 1 token in 1000 may flip


# ---- router projection with the weight split into three bf16 planes -------------------------------------------

def run_logits_split(capi, dev, x, w):
    T, H = x.shape
    E = w.shape[0]
    planes = torch.empty(3, E, H, dtype=torch.bfloat16, device=dev)
    capi.moe_router_split_weight_launch(planes, w.to(dev))
    logits = torch.full((T, E), float('nan'), device=dev)
    nbytes = capi.moe_router_logits_workspace_bytes(T, H, E)
    ws = torch.empty(nbytes, dtype=torch.uint8, device=dev) if nbytes else None
    capi.moe_router_logits_split_launch(logits, x.to(dev), planes, ws)
    torch.cuda.synchronize()
    return logits.cpu(), planes.cpu()


@pytest.mark.parametrize('shape', [(64, 7168, 256), (1, 64, 32), (100, 448, 72), (700, 1024, 256), (33, 128, 1),
                                   (130, 2048, 384), (6200, 448, 250), (12345, 64, 70),   # from here: workgroup-tiled kernel
                                   (24600, 128, 3), (24600, 192, 64), (6145, 256, 256), (6200, 320, 200),  # 1 to 5 chunks
                                   (385, 7168, 256), (1500, 2048, 130)])                  # K split 32 and 8 ways, ragged splits
def test_split_weight_logits_match_float64(capi, dev, shape):
    T, H, E = shape
    gen = torch.Generator().manual_seed(T + E + 1)
    x = torch.randn(T, H, generator=gen).bfloat16()
    w = torch.randn(E, H, generator=gen) * H ** -0.5
    w[0, :4] = torch.tensor([0.0, 1e-30, -3e38, 2.0 ** -120])
    got, planes = run_logits_split(capi, dev, x, w)
    # the planes are the oracle's, and their sum is the weight, bit for bit
    assert torch.equal(planes.view(torch.int16), moe.split_bf16x3(w).view(torch.int16))
    assert torch.equal((planes[0].float() + planes[1].float()) + planes[2].float(), w)
    w[0, 2] = 0.0                                  # (keep the reference finite)
    got, _ = run_logits_split(capi, dev, x, w)
    want = x.double() @ w.double().T
    assert torch.isfinite(got).all()
    assert ((got.double() - want).abs() <= logits_bound(x, w)).all()
    err = (got.double() - want).abs().max().item()
    ref_err = (moe.router_logits(x, w).double() - want).abs().max().item()
    assert err <= 4 * ref_err + 1e-7


def test_split_weight_logits_exact_on_integers_and_routing_chain(capi, dev):
    gen = torch.Generator().manual_seed(53)
    x = torch.randint(-8, 9, (96, 512), generator=gen).float().bfloat16()
    w = torch.randint(-8, 9, (64, 512), generator=gen).float()
    got, _ = run_logits_split(capi, dev, x, w)
    assert torch.equal(got, x.float() @ w.T)
    # hidden states -> logits -> experts at prefill size, against the oracle's chain
    T, H, E = 8192, 1024, 256
    x = torch.randn(T, H, generator=gen).bfloat16()
    w = torch.randn(E, H, generator=gen) * H ** -0.5
    bias = 0.1 * torch.randn(E, generator=gen)
    logits, _ = run_logits_split(capi, dev, x, w)
    ids, _ = run_kernel(capi, dev, logits, bias, 8, 8, 4, True, 2.5)
    want_ids, _, _ = moe.route_grouped(moe.router_logits(x, w), bias, 8, 8, 4, True, 2.5)
    assert (ids != want_ids).any(dim=1).sum().item() <= 8


def logits_of_config(capi, dev, x, w, config):
    """moe_router_logits_launcher on the kernel that `config` names; nothing is written behind the logits"""
    T, H = x.shape
    E = w.shape[0]
    x, w = x.to(dev), w.to(dev)
    nbytes = capi.moe_router_logits_workspace_bytes(T, H, E)
    ws = torch.empty(nbytes + 16, dtype=torch.uint8, device=dev)
    got = torch.full((T * E + 8,), -7.0, device=dev)
    lib, stream = capi.library(), torch.cuda.current_stream().cuda_stream
    lib.moe_router_logits_launcher(got.data_ptr(), x.data_ptr(), w.data_ptr(), ws.data_ptr(), nbytes, T, H, E, 1, config, stream)
    assert lib.cuda_agent_amd_last_status() == 0 and (got[T * E:] == -7.0).all()
    return got[:T * E].view(T, E).cpu()


def split_logits_of_config(capi, dev, x, w, config):
    T, H = x.shape
    E = w.shape[0]
    x, w = x.to(dev), w.to(dev)
    planes = torch.empty(3, E, H, dtype=torch.bfloat16, device=dev)
    capi.moe_router_split_weight_launch(planes, w)
    nbytes = capi.moe_router_logits_workspace_bytes(T, H, E)
    ws = torch.empty(nbytes + 16, dtype=torch.uint8, device=dev)
    got = torch.full((T * E + 8,), -7.0, device=dev)
    lib, stream = capi.library(), torch.cuda.current_stream().cuda_stream
    lib.moe_router_logits_split_launcher(got.data_ptr(), x.data_ptr(), planes.data_ptr(), ws.data_ptr(), nbytes, T, H, E, config, stream)
    assert lib.cuda_agent_amd_last_status() == 0 and (got[T * E:] == -7.0).all()
    return got[:T * E].view(T, E).cpu()


def check_parts(run, capi, dev, shape, config):
    """A kernel for weights in three bf16 parts, forced at a size: as close to the exact product as an fp32 evaluation, which it
    is not without the lowest part; and exact where all sums are, with weights that need all three parts"""
    T, H, E = shape
    gen = torch.Generator().manual_seed(T + H + E)
    x = torch.randn(T, H, generator=gen).bfloat16()
    w = torch.randn(E, H, generator=gen) * H ** -0.5
    got, want = run(capi, dev, x, w, config), x.double() @ w.double().T
    error = (got.double() - want).abs()
    assert (error <= logits_bound(x, w)).all()
    # (the oracle's own error as the measure, on at least 64 x 64 sums of this length: it is a maximum over random values)
    xm, wm = x, w
    if T < 64 or E < 64:
        xm, wm = torch.randn(64, H, generator=gen).bfloat16(), torch.randn(64, H, generator=gen) * H ** -0.5
    ref_err = (moe.router_logits(xm, wm).double() - xm.double() @ wm.double().T).abs().max().item()
    assert error.max().item() <= 4 * ref_err + 1e-7
    # integers of 19 bits times -1, 0 and 1, at most 31 of them a token: every sum is below 2^24
    x = torch.zeros(T, H)
    at = torch.randint(0, H, (T, 31), generator=gen)
    x.scatter_(1, at, torch.randint(-1, 2, (T, 31), generator=gen).float())
    w = torch.randint(-2 ** 19 + 1, 2 ** 19, (E, H), generator=gen).float()
    assert torch.equal(run(capi, dev, x.bfloat16(), w, config).double(), x.double() @ w.double().T)


@pytest.mark.parametrize('shape', [(1, 64, 1), (127, 128, 63), (129, 192, 65), (64, 256, 64), (257, 320, 130), (40, 7168, 8),
                                   (300, 2112, 256), (8192, 3072, 256)])    # 1 to 5 chunks a split, ragged splits, one split
def test_long_sums(capi, dev, shape):
    # the kernel whose wavefronts share K
    check_parts(logits_of_config, capi, dev, shape, 3)


@pytest.mark.parametrize('shape', [(1, 64, 1), (16, 512, 5), (17, 576, 6), (33, 3584, 256), (5, 3648, 64), (64, 7168, 257),
                                   (130, 2048, 9)])    # 1 to 112 chunks of K for 8 wavefronts of 7 in flight
def test_few_tokens_in_one_launch(capi, dev, shape):
    check_parts(split_logits_of_config, capi, dev, shape, 4)


@pytest.mark.parametrize('config', [1, 2])     # workgroups of 64 tokens x 32 experts, and of 128 x 64
@pytest.mark.parametrize('shape', [(1, 64, 32), (100, 448, 72), (33, 128, 1), (96, 512, 64), (300, 2048, 72), (129, 192, 65),
                                   (2100, 128, 130),    # one split and several, tokens and experts beyond the last tile
                                   # more chunks than are fetched ahead: 512 workgroups (four ahead) and 528 (two)
                                   (4090, 7168, 30), (4200, 7168, 30)])
def test_kernels_of_the_split_weight(capi, dev, shape, config):
    check_parts(split_logits_of_config, capi, dev, shape, config)


@pytest.mark.parametrize('config', [0, 1])
def test_more_experts_than_tiles_of_32_fit_a_grid(capi, dev, config):
    # ... go to the tiles of 64, also where the other kernel is asked for and for a single token
    check_parts(split_logits_of_config, capi, dev, (1, 64, 32 * 65535 + 1), config)


def test_bf16_parts_of_special_weights(capi, dev):
    # infinities, NaN and weights whose lower parts the matrix core would take for zero give what fp32 products give
    gen = torch.Generator().manual_seed(91)
    x = torch.randn(130, 512, generator=gen).bfloat16()
    w = torch.randn(70, 512, generator=gen)
    x[5, 100], x[7, 3] = float('inf'), float('nan')
    w[9, 50], w[11, 60], w[13, 100] = float('-inf'), float('nan'), 0.0
    w[15] = w[15].bfloat16().float()      # (parts that are zero, also beside the infinite x)
    want = torch.nn.functional.linear(x.double(), w.double())
    got = run_logits(capi, dev, x, w)
    finite = torch.isfinite(want)
    assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(got[~finite].isinf(), want[~finite].isinf())
    assert torch.equal(got[torch.isinf(want)].double(), want[torch.isinf(want)])
    assert ((got.double() - want).abs()[finite] <= logits_bound(torch.nan_to_num(x, 0, 0, 0), torch.nan_to_num(w, 0, 0, 0))[finite]).all()
    x = (torch.randn(130, 512, generator=gen) * 2.0 ** 100).bfloat16()
    w = torch.randn(70, 512, generator=gen) * 2.0 ** -130
    got = run_logits(capi, dev, x, w)
    assert ((got.double() - x.double() @ w.double().T).abs() <= logits_bound(x, w)).all()


@pytest.mark.parametrize('shape', [(64, 192, 64), (130, 512, 70), (300, 2112, 256), (4100, 448, 33)])    # one split and several
def test_bf16_parts_of_numbers_of_every_size(capi, dev, shape):
    # An expert with a weight too small for three bf16 parts, and sums that infinities turn into a NaN, get the sums of the
    # fp32 matrix cores; nothing beside them changes. Subnormal values of x count like any others
    T, H, E = shape
    gen = torch.Generator().manual_seed(T + H + E)
    x = torch.randn(T, H, generator=gen).bfloat16()
    x[3] = (torch.randn(H, generator=gen) * 2.0 ** -128).bfloat16()
    x[4] = 2.0 ** -133
    w = torch.randn(E, H, generator=gen) * 2.0 ** 60
    w[11] = 2.0 ** -110 * (1.0 + 2.0 ** -23)             # (the smallest that is the sum of its parts)
    plain = logits_of_config(capi, dev, x, w, 3)
    w0 = w.clone()
    w0[5] = torch.randn(H, generator=gen) * 2.0 ** -118
    w0[E - 1, H - 2] = 2.0 ** -149
    x2, w2 = x.clone(), w0.clone()
    x2[40, 0], x2[41, H - 1] = float('nan'), float('-inf')
    w2[7, 9] = float('inf')
    fp32 = logits_of_config(capi, dev, x2, w2, 1)
    got = logits_of_config(capi, dev, x2, w2, 3)
    want = x2.double() @ w2.double().T
    finite = torch.isfinite(want)
    assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(got[torch.isinf(want)].double(), want[torch.isinf(want)])
    assert (~finite).sum() == T + 2 * E - 2
    small = torch.zeros(T, E, dtype=torch.bool)
    small[:, [5, E - 1]] = True
    if capi.library().moe_router_logits_num_splits(T, H, E) == 1:     # (else only the splits that hold such a number)
        assert torch.equal(got[small & finite], fp32[small & finite])
    assert torch.equal(got[~small & finite], plain[~small & finite])
    # (products below 2^-126 are rounded to multiples of 2^-149)
    assert ((got.double() - want).abs()[finite] <= (logits_bound(torch.nan_to_num(x2, 0, 0, 0), w0) + H * 2.0 ** -149)[finite]).all()


def test_router_logits_rejects_bad_arguments(capi, dev):
    logits = torch.zeros(4, 32, device=dev)
    w = torch.zeros(32, 96, device=dev)
    with pytest.raises(capi.LaunchRejected):          # hidden not a multiple of 64
        capi.moe_router_logits_launch(logits, torch.zeros(4, 96, device=dev), w)
    w = torch.zeros(32, 7168, device=dev)
    with pytest.raises(capi.LaunchRejected):          # K is split for 4 tokens: scratch needed
        capi.moe_router_logits_launch(logits, torch.zeros(4, 7168, device=dev), w)
    torch.cuda.synchronize()


# ---- RMS norm fused with the activation quantiser -------------------------------------------------

@pytest.mark.parametrize('shape', [(64, 7168), (5, 128), (300, 2048), (1, 8192), (33, 384)])
@pytest.mark.parametrize('config', [0, 32])
def test_rmsnorm_quant(capi, dev, shape, config):
    R, C = shape
    gen = torch.Generator().manual_seed(R + C)
    x = (torch.randn(R, C, generator=gen) * torch.exp(torch.randn(R, 1, generator=gen))).bfloat16()
    w = (1.0 + 0.2 * torch.randn(C, generator=gen)).bfloat16()
    q = torch.empty(R, C, dtype=torch.uint8, device=dev)
    s = torch.empty(R, C // 128, device=dev)
    y = torch.empty(R, C, dtype=torch.bfloat16, device=dev)
    capi.moe_rmsnorm_quant_launch(q, s, y, x.to(dev), w.to(dev), 1e-6, config)
    torch.cuda.synchronize()
    # the normalised row: the oracle's bf16 value, or its neighbour where the fp32 sums of squares differ in the
    # last place (different order of the additions) and the value sits on a bf16 rounding boundary
    want_y = moe.rmsnorm_bf16(x, w)
    assert (y.cpu() == want_y).float().mean().item() >= 0.995
    assert ((y.cpu().float() - want_y.float()).abs() <= want_y.float().abs() * 2.0 ** -7).all()
    # the quantisation of the kernel's own y: bit-exact
    want_q, want_s = moe.quantize_groups(y.cpu().float(), pow2=config == 32)
    assert torch.equal(s.cpu(), want_s)
    assert torch.equal(q.cpu(), want_q.view(torch.uint8))
    # y is optional
    q2 = torch.empty_like(q)
    s2 = torch.empty_like(s)
    capi.moe_rmsnorm_quant_launch(q2, s2, None, x.to(dev), w.to(dev), 1e-6, config)
    torch.cuda.synchronize()
    assert torch.equal(q2, q) and torch.equal(s2, s)


@pytest.mark.parametrize('shape', [(513, 7168), (600, 2176), (1030, 128), (520, 8192), (1601, 7168), (1605, 2176), (1610, 8192),
                                   (769, 2048), (780, 1152), (577, 1024), (7700, 7168)])
def test_rmsnorm_quant_many_rows(capi, dev, shape):
    # (the last: x and the codes past the caches)
    # Above 576, 768 or 1600 rows, by their length, a workgroup has 256 lanes instead of 1024 but adds the squares in the
    # same order: the result is that of the same rows in launches of at most 300, bit for bit. (Not against the oracle's neighbouring bf16 value as
    # above: a flip of the first rounding is up to 2^-7 of the normalised value and the rounding of its product with the
    # weight can add a step of its own, which millions of values show.)
    R, C = shape
    gen = torch.Generator().manual_seed(R * 3 + C)
    x = (torch.randn(R, C, generator=gen) * torch.exp(torch.randn(R, 1, generator=gen))).bfloat16().to(dev)
    w = (1.0 + 0.2 * torch.randn(C, generator=gen)).bfloat16().to(dev)
    outs = []
    for step in (R, 300):
        q = torch.empty(R, C, dtype=torch.uint8, device=dev)
        s = torch.empty(R, C // 128, device=dev)
        y = torch.empty(R, C, dtype=torch.bfloat16, device=dev)
        for r in range(0, R, step):
            capi.moe_rmsnorm_quant_launch(q[r:r + step], s[r:r + step], y[r:r + step], x[r:r + step], w, 1e-6, 0)
        torch.cuda.synchronize()
        outs.append((q, s, y))
    for a, b in zip(*outs):
        assert torch.equal(a, b)


def test_rmsnorm_quant_golden_fixture(capi, dev):
    z = np.load(Path(__file__).parent / 'golden' / 'rmsnorm_golden.npz')
    x, w = torch.from_numpy(z['x']).bfloat16(), torch.from_numpy(z['weight']).bfloat16()
    R, C = x.shape
    q = torch.empty(R, C, dtype=torch.uint8, device=dev)
    s = torch.empty(R, C // 128, device=dev)
    y = torch.empty(R, C, dtype=torch.bfloat16, device=dev)
    capi.moe_rmsnorm_quant_launch(q, s, y, x.to(dev), w.to(dev))
    torch.cuda.synchronize()
    want = torch.from_numpy(z['y'])
    assert (y.cpu().float() == want).float().mean().item() >= 0.995
    assert ((y.cpu().float() - want).abs() <= want.abs() * 2.0 ** -7).all()


def test_rmsnorm_quant_rejects_bad_shapes(capi, dev):
    x = torch.zeros(2, 8320, dtype=torch.bfloat16, device=dev)        # more than 8192 columns
    with pytest.raises(capi.LaunchRejected):
        capi.moe_rmsnorm_quant_launch(torch.empty(2, 8320, dtype=torch.uint8, device=dev),
                                      torch.empty(2, 65, device=dev), None, x, torch.zeros(8320, dtype=torch.bfloat16, device=dev))
    torch.cuda.synchronize()
