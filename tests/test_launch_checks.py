"""The native host side of the launch helpers: what is no ordinary call is declined, launches nothing and goes on to the
checks in Python, which raise what they always raised or serve the call."""
import ctypes
import os
import re

import pytest
import torch

from oracle import gdn as ogdn


class Wrapped(torch.Tensor):
    pass


def gdn_tensors(device, gen=None):
    return [t.to(device) for t in ogdn.gdn_make_inputs(2, 4, 2, qkv_dtype=torch.bfloat16, generator=gen)]


def test_tensors_that_are_not_on_a_gpu_are_declined():
    from cuda_agent_amd import capi
    q, k, v, g, beta, state = gdn_tensors('cpu')
    o = torch.empty(2, 4, 128)
    assert capi._native.gdn_decode(o, state, q, k, v, g, beta, 0, None) == -1
    assert capi._native.topk_select(torch.zeros(1, 2, dtype=torch.int32), torch.zeros(1, 4), None, None) == -1
    assert capi._native.topk_select(None, 3, 'x', None) == -1
    with pytest.raises(ValueError, match='must be a GPU tensor'):
        capi.gdn_decode_launch(o, state, q, k, v, g, beta)
    with pytest.raises(TypeError):
        capi._native.gdn_decode(o)


@pytest.mark.gpu
def test_declined_calls_are_served_or_refused_as_before(capi, dev):
    gen = torch.Generator().manual_seed(5)
    q, k, v, g, beta, state = gdn_tensors(dev, gen)
    outs = []
    for wrap, stream in ((lambda t: t, None), (lambda t: t.as_subclass(Wrapped), None), (lambda t: t, torch.cuda.Stream()),
                         (torch.nn.Parameter, None)):
        o, s = torch.empty(2, 4, 128, device=dev), state.clone()
        torch.cuda.synchronize()
        with torch.no_grad():
            capi.gdn_decode_launch(o, s, wrap(q), k, v, g, beta, stream=stream)
        torch.cuda.synchronize()
        outs.append((o, s))
    for o, s in outs[1:]:
        assert torch.equal(o, outs[0][0]) and torch.equal(s, outs[0][1])
    o = torch.empty(2, 4, 128, device=dev)
    for bad in (dict(q=q.float()), dict(q=q[:1]), dict(v=v.transpose(1, 2)), dict(g=g.bfloat16()), dict(o=o.bfloat16())):
        args = dict(o=o, state=state, q=q, k=k, v=v, g=g, beta=beta)
        args.update(bad)
        with pytest.raises(ValueError):
            capi.gdn_decode_launch(**args)
    with pytest.raises(capi.LaunchRejected, match='gdn_decode_launcher: launch rejected'):   # head dimensions without a kernel
        capi.gdn_decode_launch(o[..., :64].contiguous(), state[..., :64].contiguous(), q, k, v[..., :64].contiguous(), g, beta)
    assert capi.library().cuda_agent_amd_last_status() == 0


# ---- the native checks against those in Python, call by call -------------------------------------------------------
# launch_checks.cpp is built once more for tensors in host memory, over launchers that write down what they are called
# with. A call that it accepts must be one that the checks in Python accept, with the same launch.

STUB = '''
#include <Python.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>
#include <sstream>
namespace c10::hip {
struct NoStream { hipStream_t stream() const { return nullptr; } };
inline NoStream noStream() { return {}; }
}
#define is_cuda is_cpu
#define getCurrentHIPStream noStream
#include "%s"
static std::string record;
template <typename... A> static void write_down(const char* name, A... a) {
    std::ostringstream s;
    s.precision(17);
    s << name;
    ((s << ' ' << a), ...);
    record = s.str();
}
extern "C" {
const char* recorded() { return record.c_str(); }
void forget() { record.clear(); }
int cuda_agent_amd_last_status() { return 0; }
%s
}
'''


@pytest.fixture(scope='module')
def stub(tmp_path_factory):
    import importlib.machinery
    import importlib.util
    import subprocess
    import sysconfig

    import torch.utils.cpp_extension as cpp_ext
    from cuda_agent_amd import PACKAGE_DIR, capi
    header = re.sub(r'/\*.*?\*/', '', (PACKAGE_DIR.parent / 'include' / 'cuda_agent_amd.h').read_text(), flags=re.S)
    launchers = []
    for name, parameters in re.findall(r'void (\w+_launcher)\(([^)]*)\);', header):
        names = [p.split()[-1].lstrip('*') for p in parameters.split(',')]
        values = [f'(void*){n}' if '*' in p else n for p, n in zip(parameters.split(','), names)]
        launchers.append(f'void {name}({parameters}) {{ write_down("{name}", {", ".join(values)}); }}')
    folder = tmp_path_factory.mktemp('launch_checks')
    source, out = folder / 'stub.cpp', folder / 'stub.so'
    source.write_text(STUB % (PACKAGE_DIR / 'launch_checks.cpp', '\n'.join(launchers)))
    torch_lib = f'{torch.__path__[0]}/lib'
    includes = [*cpp_ext.include_paths(), sysconfig.get_paths()['include'],
                (os.environ.get('ROCM_PATH') or os.environ.get('ROCM_HOME') or '/opt/rocm') + '/include']
    subprocess.run([os.environ.get('CXX', 'g++'), '-O0', '-std=c++17', '-fPIC', '-shared', '-Wl,-Bsymbolic', '-D__HIP_PLATFORM_AMD__=1', '-DUSE_ROCM=1',
                    *(f for d in dict.fromkeys(includes) for f in ('-isystem', str(d))), str(source), '-o', str(out),
                    f'-L{torch_lib}', f'-Wl,-rpath,{torch_lib}', '-lc10', '-ltorch_cpu', '-ltorch', '-ltorch_python'], check=True)
    loader = importlib.machinery.ExtensionFileLoader('launch_checks', str(out))
    native = importlib.util.module_from_spec(importlib.util.spec_from_file_location('launch_checks', out, loader=loader))
    loader.exec_module(native)
    library = ctypes.CDLL(str(out))
    library.recorded.restype = ctypes.c_char_p
    for name, (restype, argtypes) in capi.SIGNATURES.items():
        if name.endswith('_launcher'):
            getattr(library, name).restype, getattr(library, name).argtypes = restype, argtypes
    return native, library


class Spy:
    """The native functions, or with `decline` none of them, and the result of the last call."""

    def __init__(self, native, decline):
        self.native, self.decline, self.result = native, decline, None

    def __getattr__(self, name):
        def call(*args):
            self.result = -1 if self.decline else getattr(self.native, name)(*args)
            return self.result
        return call


BF16, F16, F32, F64, I32, I64, U8, E4M3 = (torch.bfloat16, torch.float16, torch.float32, torch.float64, torch.int32,
                                           torch.int64, torch.uint8, torch.float8_e4m3fn)


def zeros(dtype, *shape):
    return torch.zeros(shape, dtype=torch.uint8).to(dtype) if dtype == E4M3 else torch.zeros(shape, dtype=dtype)


def ordinary_calls():
    """helper of capi.py -> argument lists of ordinary calls, in the helper's order"""
    t = zeros
    B, H, N, k = 3, 32, 70, 40
    gates = [t(F32, B, 4), t(F32, B, 4), t(F32, 4), t(F32, 4)]
    calls = {'gdn_decode_launch': [], 'gdn_decode_fused_launch': [], 'gdn_decode_fused_norm_launch': [],
             'causal_conv1d_update_launch': []}
    for d in (BF16, F32):
        qkv = [t(F32, B, 4, 128, 128), t(d, B, 2, 128), t(d, B, 2, 128), t(d, B, 4, 128)]
        calls['gdn_decode_launch'].append([t(F32, B, 4, 128), *qkv, *gates[:2], 0, None])
        calls['gdn_decode_fused_launch'].append([t(F32, B, 4, 128), *qkv, *gates, 0, None])
        calls['gdn_decode_fused_norm_launch'].append([t(d, B, 4, 128), *qkv, *gates, t(d, B, 4, 128), t(d, 128), 1e-6, 0, None])
        conv = [t(d, B, 256, 4), t(d, B, 256), t(d, 256, 4)]
        calls['causal_conv1d_update_launch'] += [[t(d, B, 64), t(d, B, 64), t(d, B, 128), *conv, t(d, 256), 'silu', 0, None],
                                                 [None, None, t(d, B, 256), *conv, None, None, 0, None]]
    for form, row in (('', (BF16, 576)), ('_fp8', (U8, 656))):
        for d in (BF16, F32):
            head, tail = [t(d, B, H, 512), t(BF16, B, H, 576)], [t(I32, B, k), t(U8, 4096), 0.07, 0, None]
            calls.setdefault(f'sparse_mla_decode{form}_launch', []).append([*head, t(row[0], B, N, row[1]), *tail])
            for table in (t(I32, B, 5), None):
                calls.setdefault(f'sparse_mla_decode{form}_paged_launch', []).append([*head, t(row[0], 9, 16, row[1]), table, *tail])
    for lengths in (None, t(I32, B)):
        q, w = t(BF16, B, 8, 128), t(F32, B, 8)
        calls.setdefault('mla_index_scores_launch', []).append([t(F32, B, N), q, t(BF16, B, N, 128), w, lengths, 0.09, None])
        calls.setdefault('mla_index_scores_paged_launch', []).append(
            [t(F32, B, 80), q, t(BF16, 9, 16, 128), t(I32, B, 5), w, lengths, 0.09, None])
        for d in (U8, E4M3):
            q = t(d, B, 8, 128)
            calls.setdefault('mla_index_scores_fp8_launch', []).append(
                [t(F32, B, N), q, t(d, B, N, 128), t(F32, B, N), w, lengths, 0.09, None])
            calls.setdefault('mla_index_scores_fp8_paged_launch', []).append(
                [t(F32, B, 80), q, t(d, 9, 16, 128), t(F32, 9, 16), t(I32, B, 5), w, lengths, 0.09, None])
        calls.setdefault('topk_select_launch', []).append([t(I32, B, k), t(F32, B, N), lengths, None])
    for d, weight in ((BF16, U8), (F32, E4M3)):
        layer = [t(d, 3, 256), t(BF16, 3, 256), t(F32, 3, 4)]
        for name, stored in (('moe_fp8_launch', 4), ('moe_fp8_fused_shared_launch', 5)):
            calls.setdefault(name, []).append([*layer, t(weight, stored, 256, 256), t(F32, stored, 2, 2), t(weight, stored, 256, 128),
                                               t(F32, stored, 2, 1), t(U8, 4096), 2, 0, None])
        calls.setdefault('moe_router_logits_launch', []).append([t(F32, 3, 4), t(d, 3, 128), t(F32, 4, 128), t(U8, 64), None])
        calls.setdefault('moe_rmsnorm_quant_launch', []).append(
            [t(weight, 3, 256), t(F32, 3, 2), t(BF16, 3, 256) if d == BF16 else None, t(BF16, 3, 256), t(BF16, 256), 1e-6, 0, None])
    calls['moe_router_logits_split_launch'] = [[t(F32, 3, 4), t(BF16, 3, 128), t(BF16, 3, 4, 128), ws, None] for ws in (None, t(U8, 64))]
    calls['moe_route_grouped_launch'] = [[t(I32, 3, 2), t(F32, 3, 2), t(F32, 3, 8), bias, 4, 2, norm, 1.5, None]
                                         for bias, norm in ((None, True), (t(F32, 8), False))]
    return calls


def variants(value):
    """What else may be given in the place of an argument"""
    if isinstance(value, torch.Tensor):
        for dtype in (BF16, F16, F32, F64, I32, I64, U8, E4M3, torch.bool):
            if dtype != value.dtype:
                yield zeros(dtype, *value.shape)
        yield value.unsqueeze(0)
        yield value.unsqueeze(-1)
        yield value.flatten()
        for i, n in enumerate(value.shape):
            for size in (0, n - 1, n + 1, 2 * n):
                yield zeros(value.dtype, *value.shape[:i], size, *value.shape[i + 1:])
        if value.dim() > 1:
            yield value.mT
            yield torch.cat([value, value], dim=-1)[..., :value.shape[-1]]
        yield value.as_subclass(Wrapped)
        yield value[..., :1].expand(value.shape)
        yield None
    elif isinstance(value, bool):
        yield from (not value, 0, 1, 2, None)
    elif isinstance(value, int):
        yield from (value + 1, -1, True, 1.0, 2 ** 31 - 1, -2 ** 31, 2 ** 31, 2 ** 63, 2 ** 70, -2 ** 70, None, '1')
    elif isinstance(value, float):
        yield from (-value, 1, float('inf'), 1e300, 1e-300, None)
    else:
        yield from (None, 'silu', 'gelu', 0, zeros(F32, 3), zeros(U8, 16))


@pytest.mark.parametrize('helper', sorted(ordinary_calls()))
def test_what_is_accepted_launches_what_python_would(helper, stub, monkeypatch):
    from cuda_agent_amd import capi
    native, library = stub
    monkeypatch.setattr(capi, 'library', lambda: library)
    monkeypatch.setattr(capi, '_stream', lambda stream=None: 0 if stream is None else int(stream))

    def contiguous(**tensors):
        for name, tensor in tensors.items():
            capi._require(tensor.is_contiguous(), name)

    monkeypatch.setattr(capi, '_device_contiguous', contiguous)

    def call(args, decline):
        spy = Spy(native, decline)
        monkeypatch.setattr(capi, '_native', spy)
        library.forget()
        try:
            getattr(capi, helper)(*args)
            error = None
        except Exception as e:
            error = e
        return spy.result, library.recorded().decode(), error

    def check(args):
        result, launched, error = call(args, False)
        if result == -1:
            return False
        assert result == 0 and error is None and launched
        declined, want, error = call(args, True)
        assert declined == -1 and error is None and launched == want
        return True

    for args in ordinary_calls()[helper]:
        assert check(args)
        for i, value in enumerate(args):
            for other in variants(value):
                check([*args[:i], other, *args[i + 1:]])


def test_numbers_beyond_int_are_declined(stub):
    native, _ = stub
    args = ordinary_calls()['gdn_decode_launch'][0]
    for config in (2 ** 31, -2 ** 31 - 1, 2 ** 63, -2 ** 63 - 1, 2 ** 70):
        assert native.gdn_decode(*args[:7], config, None) == -1
    assert native.gdn_decode(*args[:7], -1, None) == 0


def test_the_helpers_serve_calls_without_the_native_checks(stub, monkeypatch, tmp_path):
    # only the C-ABI library built: every call goes through the checks in Python
    from cuda_agent_amd import capi
    _, library = stub
    monkeypatch.setattr(capi, 'library', lambda: library)
    monkeypatch.setattr(capi, '_stream', lambda stream=None: 0)
    monkeypatch.setattr(capi, '_device_contiguous', lambda **tensors: None)
    monkeypatch.setattr(capi, 'LAUNCH_CHECKS', tmp_path / 'launch_checks.so')
    monkeypatch.setattr(capi, '_native', capi._LoadedOnFirstUse())
    for _ in range(2):
        library.forget()
        capi.gdn_decode_launch(*ordinary_calls()['gdn_decode_launch'][0])
        assert library.recorded().startswith(b'gdn_decode_launcher')
