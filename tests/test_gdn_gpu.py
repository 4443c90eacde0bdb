"""GPU parity of the GDN decode kernel against the oracle, through the C ABI.

Tolerance (fp32 arithmetic): |a-b| <= 1e-3*|b| + 1e-3*rms(b) for output and state
(oracle.gdn.gdn_close)."""
import os
import subprocess
import sys
from pathlib import Path

import numpy as np
import pytest
import torch

from oracle import gdn

pytestmark = pytest.mark.gpu
REPO = Path(__file__).resolve().parent.parent
GOLDEN = Path(__file__).parent / 'golden' / 'gdn_decode_golden.npz'


def run_kernel(capi, dev, ins, config=0):
    q, k, v, g, beta, state = (t.to(dev) for t in ins)
    o = torch.full((state.shape[0], state.shape[1], state.shape[3]), float('nan'), device=dev)
    capi.gdn_decode_launch(o, state, q, k, v, g, beta, config=config)
    torch.cuda.synchronize()
    return o.cpu(), state.cpu()


@pytest.mark.parametrize('config', [0, 1, 2, 3])
@pytest.mark.parametrize('shape', [(1, 16, 16, torch.float32), (3, 8, 4, torch.bfloat16),
                                   (2, 6, 6, torch.bfloat16), (5, 4, 1, torch.float32)])
def test_matches_oracle(capi, dev, shape, config):
    B, Hv, Hqk, dt = shape
    gen = torch.Generator().manual_seed(100 + B)
    ins = gdn.gdn_make_inputs(B, Hv, Hqk, qkv_dtype=dt, generator=gen)
    want_o, want_s = gdn.gdn_decode_step(*ins[:5], ins[5].clone())
    o, s = run_kernel(capi, dev, ins, config)
    assert gdn.gdn_close(o, want_o) and gdn.gdn_close(s, want_s)


def test_workload_config0_fixed_seed(capi, dev):
    gen = torch.Generator().manual_seed(20250)
    ins = gdn.gdn_make_inputs(1, 16, 16, generator=gen)
    want_o, want_s = gdn.gdn_decode_step(*ins[:5], ins[5].clone())
    o, s = run_kernel(capi, dev, ins)
    assert gdn.gdn_close(o, want_o) and gdn.gdn_close(s, want_s)
    # and the reference harness's own bound
    torch.testing.assert_close(o, want_o, atol=1e-2, rtol=1e-2)


def test_golden_fixture(capi, dev):
    z = np.load(GOLDEN)
    ins = [torch.from_numpy(z[n]) for n in ('q', 'k', 'v', 'g', 'beta', 'state')]
    o, s = run_kernel(capi, dev, ins)
    assert gdn.gdn_close(o, torch.from_numpy(z['o']))
    assert gdn.gdn_close(s, torch.from_numpy(z['new_state']))


def test_several_steps_track_the_oracle(capi, dev):
    gen = torch.Generator().manual_seed(5)
    q, k, v, g, beta, state = gdn.gdn_make_inputs(2, 8, 4, qkv_dtype=torch.bfloat16, generator=gen)
    ref_state = state.clone()
    d_state = state.to(dev)
    o = torch.empty(2, 8, 128, device=dev)
    for step in range(6):
        q, k, v, g, beta, _ = gdn.gdn_make_inputs(2, 8, 4, qkv_dtype=torch.bfloat16, generator=gen)
        want_o, ref_state = gdn.gdn_decode_step(q, k, v, g, beta, ref_state)
        capi.gdn_decode_launch(o, d_state, *(t.to(dev) for t in (q, k, v, g, beta)))
        assert gdn.gdn_close(o.cpu(), want_o), step
    assert gdn.gdn_close(d_state.cpu(), ref_state)


def test_full_batched_workload_properties(capi, dev):
    """Config 1 at full size (B=256, 32/16 heads, 537 MB of state), checked through properties
    that need no CPU pass over the state: a sampled set of heads against the oracle, pure decay
    for beta = 0 and the delta-rule write for g = beta = 1."""
    B, Hv, Hqk = 256, 32, 16
    gen = torch.Generator(device=dev).manual_seed(20251)
    q = torch.randn(B, Hqk, 128, device=dev, generator=gen)
    k = torch.randn(B, Hqk, 128, device=dev, generator=gen)
    q = (q / q.norm(dim=-1, keepdim=True)).bfloat16()
    k = (k / k.norm(dim=-1, keepdim=True)).bfloat16()
    v = torch.randn(B, Hv, 128, device=dev, generator=gen).bfloat16()
    g = torch.exp(-0.5 * torch.log1p(torch.exp(torch.randn(B, Hv, device=dev, generator=gen))))
    beta = torch.sigmoid(torch.randn(B, Hv, device=dev, generator=gen))
    state = 0.02 * torch.randn(B, Hv, 128, 128, device=dev, generator=gen)
    o = torch.empty(B, Hv, 128, device=dev)

    picks = [(0, 0), (0, 31), (17, 5), (128, 16), (255, 30), (255, 31)]
    before = {p: state[p].cpu().clone() for p in picks}
    capi.gdn_decode_launch(o, state, q, k, v, g, beta)
    torch.cuda.synchronize()
    for (b, h) in picks:
        hq = h // 2
        want_o, want_s = gdn.gdn_decode_step(
            q[b, hq][None, None].cpu(), k[b, hq][None, None].cpu(), v[b, h][None, None].cpu(),
            g[b, h][None, None].cpu(), beta[b, h][None, None].cpu(), before[(b, h)][None, None])
        assert gdn.gdn_close(o[b, h].cpu()[None, None], want_o), (b, h)
        assert gdn.gdn_close(state[b, h].cpu()[None, None], want_s), (b, h)

    # beta = 0: the state is only scaled by g (bit-exact: one fp32 multiply per element)
    snap = state.clone()
    capi.gdn_decode_launch(o, state, q, k, v, g, torch.zeros_like(beta))
    torch.cuda.synchronize()
    assert torch.equal(state, snap * g[:, :, None, None])

    # g = beta = 1: probing the new state with k gives S0^T k + |k|^2 (v - S0^T k), which is v
    # up to the bf16 rounding of |k| = 1
    kf = k.float().repeat_interleave(2, 1)
    kn = (kf * kf).sum(-1, keepdim=True)
    probe0 = torch.einsum('bhij,bhi->bhj', state, kf)
    capi.gdn_decode_launch(o, state, q, k, v, torch.ones_like(g), torch.ones_like(beta))
    torch.cuda.synchronize()
    probe = torch.einsum('bhij,bhi->bhj', state, kf)
    torch.testing.assert_close(probe, probe0 + kn * (v.float() - probe0), rtol=1e-4, atol=1e-4)
    assert (probe - v.float()).abs().max().item() < 0.1


@pytest.mark.parametrize('ws_config', ['0', '1'])
def test_workspace_verification_flow(ws_config):
    """`python3 -m utils.verification` from inside the workspace, as its user runs it."""
    ws = REPO / 'cuda-agent_amd' / 'workspaces' / 'gdn_decode'
    assert (ws / 'cuda_extension.so').exists(), 'workspace extension not built'
    env = dict(os.environ, GDN_CONFIG=ws_config)
    out = subprocess.run([sys.executable, '-m', 'utils.verification'], cwd=ws, env=env,
                         capture_output=True, text=True, timeout=600)
    assert out.returncode == 0, out.stdout + out.stderr
    assert '[PASS] check 5/5' in out.stdout and '[PASS] verify success' in out.stdout


def test_workspace_rejects_bad_inputs(dev):
    ws = REPO / 'cuda-agent_amd' / 'workspaces' / 'gdn_decode'
    code = (
        "import torch, cuda_extension as e\n"
        "d='cuda:0'\n"
        "q=torch.zeros(1,2,128,device=d);v=torch.zeros(1,2,128,device=d);g=torch.ones(1,2,device=d)\n"
        "s=torch.zeros(1,2,128,128,device=d)\n"
        "o,s2=e.gdn_decode_forward(q,q,v,g,g,s,0); assert s2.data_ptr()==s.data_ptr() and o.shape==(1,2,128)\n"
        "for bad in [lambda: e.gdn_decode_forward(q.cpu(),q,v,g,g,s,0),\n"
        "            lambda: e.gdn_decode_forward(q.half(),q.half(),v.half(),g,g,s,0),\n"
        "            lambda: e.gdn_decode_forward(q,q,v,g,g,s[:,:,:64].contiguous(),0),\n"
        "            lambda: e.gdn_decode_forward(q,q,v,g,g,s.transpose(2,3),0)]:\n"
        "    try: bad(); raise SystemExit('accepted a bad input')\n"
        "    except RuntimeError: pass\n"
        "print('ok')\n")
    out = subprocess.run([sys.executable, '-c', code], cwd=ws, capture_output=True, text=True, timeout=300)
    assert out.returncode == 0 and 'ok' in out.stdout, out.stdout + out.stderr


# ---- fused pre-step (L2 normalisation of q/k and gates inside the kernel) -------------------------

FUSED_GOLDEN = Path(__file__).parent / 'golden' / 'gdn_fused_golden.npz'


def run_fused(capi, dev, ins, config=0):
    qr, kr, v, a, b, a_log, dt_bias, state = (t.to(dev) for t in ins)
    o = torch.full((state.shape[0], state.shape[1], state.shape[3]), float('nan'), device=dev)
    capi.gdn_decode_fused_launch(o, state, qr, kr, v, a, b, a_log, dt_bias, config=config)
    torch.cuda.synchronize()
    return o.cpu(), state.cpu()


@pytest.mark.parametrize('config', [0, 1, 3, 9])
@pytest.mark.parametrize('shape', [(1, 16, 16, torch.float32), (3, 8, 4, torch.bfloat16), (5, 4, 1, torch.float32)])
def test_fused_matches_oracle(capi, dev, shape, config):
    B, Hv, Hqk, dt = shape
    gen = torch.Generator().manual_seed(300 + B)
    ins = gdn.gdn_make_raw_inputs(B, Hv, Hqk, qkv_dtype=dt, generator=gen)
    want_o, want_s = gdn.gdn_decode_fused_step(*ins[:7], ins[7].clone())
    o, s = run_fused(capi, dev, ins, config)
    assert gdn.gdn_close(o, want_o) and gdn.gdn_close(s, want_s)


@pytest.mark.parametrize('dtype', [torch.float32, torch.bfloat16])
@pytest.mark.parametrize('batch', [48, 49, 64, 65, 80, 81, 96, 97])
def test_sums_by_shuffles_are_the_same_sums(capi, dev, batch, dtype):
    # With 4 heads: the edges of the sizes (193 or 257 to 320 heads of all requests, 384 of the plain step) whose sums go through the LDS
    # crossbar. A request's result is the oracle's, and that of a call with few requests bit for bit
    gen = torch.Generator().manual_seed(batch)
    for make, run, step in ((gdn.gdn_make_inputs, run_kernel, gdn.gdn_decode_step),
                            (gdn.gdn_make_raw_inputs, run_fused, gdn.gdn_decode_fused_step)):
        ins = make(batch, 4, 2, qkv_dtype=dtype, generator=gen)
        o, s = run(capi, dev, ins)
        want_o, want_s = step(*ins[:-1], ins[-1].clone())
        assert gdn.gdn_close(o, want_o) and gdn.gdn_close(s, want_s)
        parts = [run(capi, dev, [t[at:at + 24] if t.shape[0] == batch else t for t in ins]) for at in range(0, batch, 24)]
        assert torch.equal(o, torch.cat([p[0] for p in parts])) and torch.equal(s, torch.cat([p[1] for p in parts]))


def test_fused_golden_fixture(capi, dev):
    z = np.load(FUSED_GOLDEN)
    ins = [torch.from_numpy(z[n]) for n in ('q', 'k', 'v', 'a', 'b', 'a_log', 'dt_bias', 'state')]
    o, s = run_fused(capi, dev, ins)
    assert gdn.gdn_close(o, torch.from_numpy(z['o'])) and gdn.gdn_close(s, torch.from_numpy(z['new_state']))


def test_fused_equals_unfused_on_prestepped_inputs(capi, dev):
    gen = torch.Generator().manual_seed(31)
    ins = gdn.gdn_make_raw_inputs(4, 8, 4, generator=gen)
    qn, kn, g, beta = gdn.gdn_prestep(*ins[:2], *ins[3:7])
    o1, s1 = run_fused(capi, dev, ins)
    o2, s2 = run_kernel(capi, dev, [qn, kn, ins[2], g, beta, ins[7]])
    assert gdn.gdn_close(o1, o2) and gdn.gdn_close(s1, s2)


def test_fused_full_workload_shape(capi, dev):
    # configs[1] sizes; the pre-step must not cost bandwidth: compare with the unfused kernel's result
    gen = torch.Generator().manual_seed(32)
    ins = gdn.gdn_make_raw_inputs(256, 32, 16, qkv_dtype=torch.bfloat16, generator=gen)
    qn, kn, g, beta = gdn.gdn_prestep(*ins[:2], *ins[3:7])
    o1, s1 = run_fused(capi, dev, ins)
    want_o, want_s = gdn.gdn_decode_step(qn.to(dev), kn.to(dev), ins[2].to(dev), g.to(dev), beta.to(dev),
                                         ins[7].to(dev))
    assert gdn.gdn_close(o1, want_o.cpu()) and gdn.gdn_close(s1, want_s.cpu())


# ---- the fused step with the gated RMS normalisation of its read-out ------------------------------

def run_fused_norm(capi, dev, ins, z, norm_w, eps=1e-6):
    q, k, v, a, b, a_log, dt_bias, state = (t.to(dev) for t in ins)
    s = state.clone()
    out = torch.full(v.shape, float('nan'), dtype=v.dtype, device=dev)
    capi.gdn_decode_fused_norm_launch(out, s, q, k, v, a, b, a_log, dt_bias, z.to(dev), norm_w.to(dev), eps)
    torch.cuda.synchronize()
    return out.cpu(), s.cpu()


@pytest.mark.parametrize('shape', [(2, 4, 2, torch.float32), (3, 8, 4, torch.bfloat16), (1, 16, 16, torch.float32),
                                   (64, 32, 16, torch.bfloat16)])
def test_fused_norm_matches_oracle(capi, dev, shape):
    B, Hv, Hqk, dt = shape
    gen = torch.Generator().manual_seed(400 + B)
    ins = gdn.gdn_make_raw_inputs(B, Hv, Hqk, qkv_dtype=dt, generator=gen)
    z = (torch.randn(B, Hv, 128, generator=gen) * 2).to(dt)
    norm_w = (1.0 + 0.1 * torch.randn(128, generator=gen)).to(dt)
    want, want_s = gdn.gdn_decode_fused_norm_step(*ins[:7], ins[7].clone(), z, norm_w)
    out, s = run_fused_norm(capi, dev, ins, z, norm_w)
    assert gdn.gdn_close(s, want_s)
    assert out.dtype == dt
    if dt == torch.float32:
        assert gdn.gdn_close(out, want)
    else:
        # bf16 output: the oracle's value or its bf16 neighbour where the fp32 results straddle a rounding boundary
        a_, b_ = out.float(), want.float()
        assert ((a_ - b_).abs() <= torch.maximum(a_.abs(), b_.abs()) * 2.0 ** -7 + 1e-3 * b_.abs().max()).all()
        assert (out == want).float().mean() >= 0.97
    # the state is the plain fused step's, bit for bit, when that runs with the same tiling (config 9: one
    # workgroup of 1024 lanes per head); the normalisation only touches the output
    _, s_plain = run_fused(capi, dev, ins, 9)
    assert torch.equal(s, s_plain)


def test_fused_norm_equals_norm_of_the_fused_read_out(capi, dev):
    gen = torch.Generator().manual_seed(45)
    ins = gdn.gdn_make_raw_inputs(4, 8, 4, generator=gen)
    z = torch.randn(4, 8, 128, generator=gen)
    norm_w = 1.0 + 0.1 * torch.randn(128, generator=gen)
    o, _ = run_fused(capi, dev, ins)
    out, _ = run_fused_norm(capi, dev, ins, z, norm_w)
    torch.testing.assert_close(out, gdn.gated_rmsnorm(o, z, norm_w), rtol=2e-5, atol=1e-6)


def test_fused_norm_golden_fixture(capi, dev):
    # the recurrence from the fused golden fixture, then the third-party norm module's own fixture shapes the norm
    zf = np.load(FUSED_GOLDEN)
    ins = [torch.from_numpy(zf[n]) for n in ('q', 'k', 'v', 'a', 'b', 'a_log', 'dt_bias', 'state')]
    g = np.load(FUSED_GOLDEN.with_name('gated_rmsnorm_golden.npz'))
    B, Hv = ins[2].shape[:2]
    gen = torch.Generator().manual_seed(46)
    z = torch.randn(B, Hv, 128, generator=gen)
    norm_w = torch.from_numpy(g['weight'])
    out, s = run_fused_norm(capi, dev, ins, z, norm_w)
    want = gdn.gated_rmsnorm(torch.from_numpy(zf['o']), z, norm_w)
    assert gdn.gdn_close(out, want) and gdn.gdn_close(s, torch.from_numpy(zf['new_state']))
