"""Host logic on the CPU: the GradientMaker API, schedules, the hook engine and the K-FAC
orchestration, with the kernel entry points replaced by oracle-backed stand-ins
(tests/cpu_backend.py).  Also checks that the C-ABI library loads and exports every declared symbol
and that the product refuses CPU tensors."""
import contextlib
import copy
import os

import numpy as np
import pytest
import torch
import torch.nn as nn
import torch.nn.functional as F

import asdl_amd
from asdl_amd import (PreconditioningConfig, KfacGradientMaker, GradientMaker, FisherConfig, get_fisher_maker,
                      get_update_schedule, SHAPE_KRON, FISHER_EMP, FISHER_MC, FISHER_EXACT, LOSS_CROSS_ENTROPY, LOSS_MSE)
from conftest import GOLDEN
from models_small import GOLDEN_KFAC, get_mlp, get_cnn, get_tied_mlp
import cpu_backend


def relerr(a, b):
    return float((a.double() - b.double()).norm() / b.double().norm().clamp_min(1e-300))


def grad_close(got, ref, tol):
    """Relative error below tol, or both essentially zero (a bias in front of a normalisation layer has an
    exactly zero gradient; what is left of it in fp32 is rounding noise)."""
    ref = ref.double()
    got = got.detach().double().cpu()
    if float(ref.norm()) < 1e-6:
        return float((got - ref).norm()) < 1e-5
    return float((got - ref).norm() / ref.norm()) < tol


# ------------------------------------------------------------------ library / boundary
def test_library_loads_and_exports_every_declared_symbol():
    from asdl_amd import _lib
    lib = _lib.load()
    declared = _lib.declared_symbols()
    assert len(declared) >= 12
    for name in declared:
        assert hasattr(lib, name), f'{name} is declared in include/asdl_amd.h but not exported'
        assert name in _lib._SIGNATURES, f'{name} has no ctypes signature'
    assert lib.ak_version() >= 100
    assert b'workspace' in lib.ak_error_string(-2)


def test_no_hot_kernel_spills_registers():
    """asdl_amd.build writes the compiler's resource figures of every kernel next to the library.  The matrix-core
    kernels keep their accumulators in registers for the whole k-loop: scratch memory (a spill) in one of them costs
    a factor of two and more (it happened to the 256-wide gathered SYRK tile after an epilogue change), so none is
    allowed outside the short list of kernels that have always had a few bytes."""
    report = os.path.join(os.path.dirname(asdl_amd.__file__), 'lib', 'kernel_resources.txt')
    if not os.path.exists(report):
        pytest.skip('no kernel_resources.txt: the library was not built by asdl_amd.build in this tree')
    allowed = {'conv_patch_syrk_kernel': 16, 'conv_syrk_kernel': 96}        # bytes per lane
    rows = [l.split() for l in open(report) if l.strip() and not l.startswith('#')]
    assert len(rows) > 100
    spilled = []
    for src, name, vgprs, agprs, scratch, occupancy, lds in rows:
        limit = max([v for k, v in allowed.items() if k in name] or [0])
        if int(scratch) > limit:
            spilled.append((src, name, int(scratch)))
    assert not spilled, spilled


@pytest.fixture(scope='module')
def assembly(tmp_path_factory):
    """The instructions of every kernel of the built library, {name: [text]}."""
    import shutil
    import subprocess
    from asdl_amd import _lib
    objdump = '/opt/rocm/llvm/bin/llvm-objdump'
    if not os.path.exists(objdump):
        pytest.skip('no llvm-objdump')
    where = tmp_path_factory.mktemp('assembly')
    copy = shutil.copy(_lib.LIB_PATH, where / 'lib.so')
    subprocess.run([objdump, '--offloading', str(copy)], cwd=where, check=True, capture_output=True)
    kernels = {}
    for i, obj in enumerate(sorted(where.glob('lib.so.*gfx950'))):
        text = subprocess.run([objdump, '-d', '--no-show-raw-insn', '--no-leading-addr', str(obj)], check=True, capture_output=True, text=True).stdout
        for line in text.splitlines():
            line = line.split('//')[0].strip()
            if line.endswith('>:'):
                lines = kernels.setdefault(f'{line[1:-2]} {i}', [])
            elif line and not line.endswith(':') and 'file format' not in line:
                lines.append(line)
    return kernels


def test_loads_to_the_lds_wait_for_descriptors_from_vector_instructions(assembly):
    """A vector memory instruction may read a scalar register five wait states after a vector instruction (v_readfirstlane) wrote it.
    The compiler keeps that distance for its own loads, not for the inline assembly of load_to_lds(): in the assembly of the library
    as it is built no descriptor of such a load is younger, along the instructions in front of it."""
    import re
    loads, young = 0, []
    for kernel, lines in assembly.items():
        for at, line in enumerate(lines):
            if not (line.startswith('buffer_load') and line.endswith(' lds')):
                continue
            loads += 1
            low, high = map(int, re.search(r' s\[(\d+):(\d+)\]', line).groups())
            states = 0
            for earlier in reversed(lines[max(0, at - 5):at]):
                op, *operands = earlier.replace(',', ' ').split()
                if op == 's_nop':
                    states += int(operands[0], 0)
                elif op.startswith('v_') and states < 5:
                    m = re.fullmatch(r's(\d+)|s\[(\d+):(\d+)\]', operands[0])
                    if m:
                        first = int(m.group(1) or m.group(2))
                        if first <= high and int(m.group(3) or first) >= low:
                            young.append((kernel[:60], line, earlier, states))
                states += 1
    assert loads > 100
    assert not young, young


def test_chain_of_the_grouped_inverses_has_no_flat_accesses(assembly):
    """Its tiles come from the matrices or from the work matrix: both are global memory, and the kernel says so."""
    chain = [lines for name, lines in assembly.items() if 'cg_chain_kernel' in name]
    assert len(chain) == 1 and any(l.startswith('global_store') for l in chain[0])
    assert not [l for l in chain[0] if l.startswith('flat_')]


def test_kernels_that_run_beside_the_framework_hold_their_cus():
    """The kernels of the grouped inverses with 16-bit matrix instructions run on side streams.  A work group of theirs has all 512 vector
    registers of its CU's lanes, by blocks of 8 a wave, so that no wave of another kernel runs there."""
    report = os.path.join(os.path.dirname(asdl_amd.__file__), 'lib', 'kernel_resources.txt')
    if not os.path.exists(report):
        pytest.skip('no kernel_resources.txt: the library was not built by asdl_amd.build in this tree')
    rows = [l.split() for l in open(report) if l.startswith('chol_group.hip')]
    beside = {'cg_sweep_kernel': 1024, 'cg_chain_kernel': 1024, 'cg_copy_in_kernel': 0, 'cg_scale_kernel': 0, 'cg_out_kernel': 0}      # 0: no matrix instruction
    found = {k: r for k in beside for r in rows if k in r[1]}
    assert sorted(found) == sorted(beside) and sum('cg_' in r[1] for r in rows) == len(beside)
    for name, threads in beside.items():
        registers = (int(found[name][2]) + int(found[name][3]) + 7) // 8 * 8
        assert threads == 0 or threads // 64 // 4 * registers == 512, found[name]


def test_root_workspace_of_a_call_over_all_sizes_is_below_that_of_its_largest_group():
    """A call takes the roots of all sizes at once, so its workspace is a sum.  For a twelve-layer decoder of 768 columns it has to stay
    below the bound for the largest group alone, which holds for any power."""
    import ctypes
    from asdl_amd import _lib
    lib = _lib.load()
    groups = [(768, 61), (2304, 12), (3072, 24), (1024, 1)]
    count = len(groups)
    n, batch, p = (ctypes.c_int64 * count)(*(g[0] for g in groups)), (ctypes.c_int * count)(*(g[1] for g in groups)), (ctypes.c_int * count)(*[4] * count)
    need = lib.ak_inv_root_group_ws_bytes(n, batch, p, 1e-6, count)
    assert 0 < need < lib.ak_inv_root_ws_bytes(3072, 24), need
    for n1, b1, p1, eps in ((3072, 24, 4, 1e-6), (3072, 24, 4, 0.0), (600, 3, 7, 1e-6), (130, 2, 11, 1e-6), (2, 1, 1, 1e-6)):
        one = lib.ak_inv_root_group_ws_bytes(ctypes.byref(ctypes.c_int64(n1)), ctypes.byref(ctypes.c_int(b1)), ctypes.byref(ctypes.c_int(p1)), eps, 1)
        assert 0 < one <= lib.ak_inv_root_ws_bytes(n1, b1)
    assert lib.ak_inv_root_ws_bytes(40000, 1) > 4 * 40000 ** 2 and lib.ak_inv_root_ws_bytes((1 << 20) + 1, 1) == 0      # sizes taken


def test_plan_of_the_grouped_inverse_says_how_long_it_takes():
    """The library's own estimate, by which it chose the sequence: it grows with the sizes on both sides of the choice, and lies near
    what was measured (206, 284, 757 microseconds for the first three)."""
    import ctypes
    from asdl_amd import _lib
    lib = _lib.load()

    def estimate(dims):
        arr = (ctypes.c_int64 * len(dims))(*dims)
        plan = ctypes.create_string_buffer(lib.ak_chol_group_plan_bytes(arr, len(dims)))
        assert lib.ak_chol_group_plan(arr, len(dims), plan, len(plan)) == 0
        return lib.ak_chol_group_plan_us(plan)
    for dims, measured in (((784, 512, 512, 512, 512, 10), 206), ((1153, 512), 284), ((2048, 2048), 757)):
        assert 0.7 * measured < estimate(dims) < 1.3 * measured, (dims, estimate(dims))
    assert estimate((4096, 4096)) > estimate((2048,) * 4) > estimate((2048, 2048)) > estimate((128,)) > 0
    assert lib.ak_chol_group_plan_us(ctypes.create_string_buffer(256)) < 0


def test_grouped_inverse_plans_do_not_depend_on_the_queries_before():
    import ctypes
    from asdl_amd import _lib
    lib = _lib.load()

    def plan_of(dims, others=()):
        arr = (ctypes.c_int64 * len(dims))(*dims)
        plan = ctypes.create_string_buffer(lib.ak_chol_group_plan_bytes(arr, len(dims)))
        for other in others:
            lib.ak_chol_group_ws_bytes((ctypes.c_int64 * len(other))(*other), len(other))
        assert lib.ak_chol_group_plan(arr, len(dims), plan, len(plan)) == 0
        return plan.raw, lib.ak_chol_group_ws_bytes(arr, len(dims))
    for dims in ((784, 512, 10), (1100,) * 24, (4225,)):
        assert plan_of(dims) == plan_of(dims) == plan_of(dims, others=((300,), dims[:-1] + (9,)))


@pytest.mark.parametrize('dims', [(2817,), (2944,), (3072,), (3073,), (3500,), (2600, 2304, 2048, 1500, 700, 600), (2892, 2892, 1400, 700, 300, 200),
                                  (1601, 2836, 542, 176, 670, 81, 44, 19)])
def test_inverses_that_the_sweep_can_take_stay_with_its_accuracy(dims):
    """One launch per block of 128 columns: the block sweep, whose sums round least (the chain's errors on rank-deficient factors are
    two to three times larger), and whose workspace is the tiles of the triangles and two columns of them."""
    import ctypes
    from asdl_amd import _lib
    lib = _lib.load()
    arr = (ctypes.c_int64 * len(dims))(*dims)
    plan = ctypes.create_string_buffer(lib.ak_chol_group_plan_bytes(arr, len(dims)))
    assert lib.ak_chol_group_plan(arr, len(dims), plan, len(plan)) == 0
    blocks = [(d + 127) // 128 for d in dims]
    assert lib.ak_chol_group_plan_launches(plan) == max(blocks) + 1
    assert lib.ak_chol_group_ws_bytes(arr, len(dims)) == 4 * 128 * 128 * sum(n * (n + 1) // 2 + 2 * n + 2 for n in blocks)


def test_factor_workspaces_are_for_kernels_that_may_run():
    """fp32 rows beyond the wave kernel's rule, bf16 rows and statistics in a fixed order do not ask for its partial sums."""
    from asdl_amd import _lib, kernels
    lib = _lib.load()
    f32, bf16, ordered = 0, 1, kernels.AK_F32_IN_ORDER
    assert lib.ak_syrk_tn_ws_bytes_of(f32, 8192, 4096) == lib.ak_syrk_tn_ws_bytes_of(bf16, 8192, 4096) == lib.ak_syrk_tn_ws_bytes(8192, 4096) == 0
    assert lib.ak_conv_syrk_ws_bytes_of(ordered, 1, 4096, 1, 16384, 1, 1, 1, 1, 0, 0) == 0
    assert lib.ak_conv_syrk_ws_bytes_of(bf16, 1, 4096, 1, 16384, 1, 1, 1, 1, 0, 0) == 0
    for M, d in ((128, 784), (1000, 1021), (70000, 40), (4096, 700), (3136, 2048)):       # the query for all types holds each
        assert lib.ak_syrk_tn_ws_bytes(M, d) >= max(lib.ak_syrk_tn_ws_bytes_of(t, M, d) for t in (f32, bf16, ordered))
        assert lib.ak_syrk_tn_ws_bytes_of(ordered, M, d) <= lib.ak_syrk_tn_ws_bytes_of(f32, M, d)
    for conv in ((128, 64, 32, 32, 3, 3, 1, 1, 1, 1), (128, 64, 32, 32, 1, 1, 1, 1, 0, 0), (128, 256, 8, 8, 1, 1, 2, 2, 0, 0), (64, 48, 20, 20, 3, 3, 1, 1, 1, 1),
                 (64, 3, 32, 32, 3, 3, 1, 1, 1, 1)):
        each = [lib.ak_conv_syrk_ws_bytes_of(t, *conv) for t in (f32, bf16, ordered)]
        assert lib.ak_conv_syrk_ws_bytes(*conv) >= max(each) > 0


@pytest.mark.parametrize('N,C,H,k,s,p,planes', [
    # many columns and few positions, where the planes' partial tiles alone take longer: us measured on the fp32 kernel and on planes
    (16, 1024, 4, 3, 2, 1, False),       # 173, 243
    (2, 1600, 9, 3, 2, 1, False),        # 434, 555
    (4, 1696, 7, 3, 2, 1, False),        # 503, 636
    (4, 2048, 4, 3, 2, 1, False),        # 719, 840
    (16, 2048, 4, 3, 2, 1, False),       # 778, 891
    (8, 300, 7, 3, 1, 1, False),         # 60, 64
    # and where the products do
    (64, 1024, 4, 3, 2, 1, True),        # 354, 301
    (64, 2048, 4, 3, 2, 1, True),        # 1410, 1137
    (128, 2048, 8, 3, 2, 1, True),       # 7931, 3891
    (64, 512, 4, 3, 2, 1, True),         # 99, 80
    (128, 256, 8, 3, 2, 1, True),        # 163, 97
    (128, 128, 8, 3, 2, 1, True),        # 61, 44
    (32, 64, 32, 3, 2, 1, True),         # 72, 48
    (8, 600, 7, 5, 1, 2, True),          # 1296, 942
])
def test_windows_of_fp32_inputs_go_to_the_faster_kernel(N, C, H, k, s, p, planes):
    from asdl_amd import _lib
    lib = _lib.load()
    need = lib.ak_conv_syrk_planes_ws_bytes(N, C, H, H, k, k, s, s, p, p)
    assert (need > 0) == planes
    # the query for a call holds it, and the partial tiles stay below half the padded factor and a round of splits
    assert lib.ak_conv_syrk_ws_bytes_of(0, N, C, H, H, k, k, s, s, p, p) >= need
    frame, padded = ((H + 2 * p - k) // s * s + k) ** 2, (C + 31) // 32 * 32
    tiles = -(-padded * k * k // 128)
    assert need <= N * frame * 6 * padded + 256 + (512 + tiles * (tiles + 1) // 2) * 65536


def test_small_module_preconditioning_leaves_sizes_beyond_its_own_to_the_other_paths():
    """The row matrices of the swift variant have inverses of more than 32768 columns.  The two-launch form declines them, before it
    launches anything, instead of refusing the call."""
    import ctypes
    from asdl_amd import _lib, kernels
    lib = _lib.load()

    def ask(items, units, only_if_faster):
        return lib.ak_kron_precond_deep((ctypes.c_int64 * len(items))(*items), len(items) // 6, (ctypes.c_int64 * len(units))(*units),
                                        len(units) // 4, 1.0, 0, 0, only_if_faster, 0, 0, 0)
    small = [16, 16, 16, 0, 8, 8]
    for only in (0, 1):
        assert ask(small + [16, 16, 16, 0, 40000, 8], [], only) == kernels.AK_ERR_UNSUPPORTED
        assert ask([16, 16, 16, 0, 8, (1 << 20) + 1], [], only) == kernels.AK_ERR_UNSUPPORTED
        assert ask([], [16, 16, 16, (1 << 24) + 1], only) == kernels.AK_ERR_UNSUPPORTED
    assert ask([16, 16, 0, 0, 8, 8], [], 0) == -1 and ask([], [16, 16, 16, 0], 0) == -1       # (no gradient, no features: errors)


def test_product_refuses_cpu_tensors():
    from asdl_amd import kernels
    with pytest.raises(RuntimeError, match='ROCm device'):
        kernels.syrk_tn(torch.randn(4, 4))
    with pytest.raises(RuntimeError, match='ROCm device'):
        kernels.conv_syrk(torch.randn(1, 2, 4, 4), (3, 3), (1, 1), (1, 1))
    with pytest.raises(RuntimeError, match='ROCm device'):
        asdl_amd.cholesky_inv(torch.eye(3), 0.1)
    model = get_mlp()
    gm = KfacGradientMaker(model, PreconditioningConfig(data_size=2, damping=1e-2), fisher_type=FISHER_EMP)
    x, t = torch.randn(2, 5), torch.randint(4, (2,))
    gm.setup_loss_call(F.cross_entropy, gm.setup_model_call(model, x), t)
    with pytest.raises(RuntimeError, match='ROCm device'):
        gm.forward_and_backward()


# ------------------------------------------------------------------ GradientMaker API (test/grad_maker/test_grad_maker.py)
class _Net(nn.Module):
    def __init__(self):
        super().__init__()
        self.model = get_mlp()

    def forward(self, inputs, targets=None, flip=False):
        logits = self.model(inputs)
        if targets is not None:
            loss = F.cross_entropy(logits, targets)
            return (loss, logits) if flip else (logits, loss)
        return logits


def _vanilla(model, x, t):
    model.zero_grad(set_to_none=True)
    loss = F.cross_entropy(model(x), t)
    loss.backward()
    return loss, [p.grad.clone() for p in model.parameters()]


def test_grad_maker_matches_vanilla_autograd_for_every_calling_style():
    torch.manual_seed(0)
    model = _Net()
    x, t = torch.randn(4, 5), torch.randint(4, (4,))
    ref_loss, ref_grads = _vanilla(model, x, t)
    gm = GradientMaker(model)

    def check(loss):
        torch.testing.assert_close(loss, ref_loss)
        for p, g in zip(model.parameters(), ref_grads):
            torch.testing.assert_close(p.grad, g)

    model.zero_grad(set_to_none=True)
    dummy_y = gm.setup_model_call(model, x)
    gm.setup_loss_call(F.cross_entropy, dummy_y, t)
    y, loss = gm.forward_and_backward()
    check(loss)
    torch.testing.assert_close(y, model(x))

    for flip, idx in [(False, 1), (True, 0)]:
        model.zero_grad(set_to_none=True)
        gm_repr = GradientMaker(model)
        dummy_y = gm_repr.setup_model_call(model, x, targets=t, flip=flip)
        gm_repr.setup_loss_repr(dummy_y[idx])
        y, loss = gm_repr.forward_and_backward()
        check(loss)
        # a registered loss function wins over a loss expression (asdl/grad_maker.py:272-281)
        gm_repr.setup_loss_call(lambda out: out[idx] * 2, dummy_y)
        assert torch.allclose(gm_repr.forward_and_backward()[1], ref_loss * 2)

    # delegation: the other maker runs what was registered here, results land in both
    model.zero_grad(set_to_none=True)
    other = GradientMaker(model)
    y, loss = gm.delegate_forward_and_backward(other)
    check(loss)
    assert other.loss is gm.loss and other.model_output is gm.model_output

    with pytest.raises(TypeError):
        gm.setup_loss_repr('not a dummy')
    with pytest.raises(ValueError):
        GradientMaker(model).forward_and_backward()


def test_dummy_object_replays_attribute_item_and_call():
    lin = nn.Linear(5, 3)
    assert asdl_amd.DummyObject().weight[0].numel().eval(lin) == 5
    d = asdl_amd.DummyObject()
    assert d['a'][1].eval({'a': [1, 2]}) == 2
    # placeholders among the arguments of a recorded call are evaluated on the same base value
    base = {'f': lambda a, b=0: 10 * a + b, 'x': 3, 'y': 4}
    assert d['f'](d['x'], b=d['y']).eval(base) == 34
    assert d['a'].eval({'a': 1}) == 1 and d.eval(7) == 7        # d itself was not changed by the longer paths


def test_loss_reduction_override_for_functions_and_modules():
    """A maker that names a reduction passes it as a keyword to loss functions and sets (then restores) the
    attribute of loss modules; a loss without the option is refused (asdl/grad_maker.py:283-300)."""
    class Summed(GradientMaker):
        _loss_reduction = 'sum'

    torch.manual_seed(0)
    model = _Net()
    x, t = torch.randn(4, 5), torch.randint(4, (4,))
    expected = F.cross_entropy(model(x), t, reduction='sum')
    gm = Summed(model)
    gm.setup_loss_call(F.cross_entropy, gm.setup_model_call(model, x), t, reduction='mean')
    torch.testing.assert_close(gm.forward_and_backward()[1], expected)
    crit = nn.CrossEntropyLoss()
    gm.setup_loss_call(crit, gm.setup_model_call(model, x), t)
    torch.testing.assert_close(gm.forward_and_backward()[1], expected)
    assert crit.reduction == 'mean'
    gm.setup_loss_call(lambda y, t: F.cross_entropy(y, t), gm.setup_model_call(model, x), t)
    with pytest.raises(AttributeError):
        gm.forward_and_backward()


# ------------------------------------------------------------------ schedules
def test_update_schedule_and_intervals():
    s = get_update_schedule(10, update_ratio=0.5)
    assert len(s) == 10 and sum(s) == 5 and s[0]
    s = get_update_schedule(10, update_ratio=0.5, warmup_ratio=0.2)
    assert s[:2] == [True, True] and sum(s) == 5
    assert get_update_schedule(4, 1.0) == [True] * 4
    assert get_update_schedule(6, 0.5, interval_type='step') == [True] * 3 + [False] * 3
    # vectors worked out by hand from asdl/precondition/prec_grad_maker.py:204-254
    T_, F_ = True, False
    assert get_update_schedule(10, 0.5) == [T_, F_] * 5
    assert get_update_schedule(10, 0.3) == [T_, F_, F_, T_, F_, F_, T_, F_, F_, F_]      # the 4th multiple of 3 is over budget
    assert get_update_schedule(10, 0.5, 0.2) == [T_, T_, T_, F_, T_, F_, T_, F_, F_, F_]
    assert get_update_schedule(10, 0.5, 0.2, reverse=True) == [T_, T_, T_, F_, T_, F_, T_, F_, F_, F_][::-1]
    linear = get_update_schedule(20, 0.25, interval_type='linear')         # gaps 0, 2, 4, 6
    assert [i for i, f in enumerate(linear) if f] == [0, 1, 4, 9, 16] and len(linear) == 20
    with pytest.raises(ValueError):
        get_update_schedule(10, 0.5, interval_type='linear')               # gaps 0, 1, 2, 3 end at step 11 of 10
    with pytest.raises(ZeroDivisionError):
        get_update_schedule(10, 0.2, interval_type='linear')               # two updates: n (n - 1) = 0
    with pytest.raises(ValueError):
        get_update_schedule(10, 0.2, warmup_ratio=0.5)
    with pytest.raises(ValueError):
        get_update_schedule(10, 0.5, interval_type='quadratic')
    with pytest.raises(ValueError):
        get_update_schedule(0)
    with pytest.raises(ValueError):
        get_update_schedule(10, 1.5)
    gm = KfacGradientMaker(get_mlp(), PreconditioningConfig(data_size=1, preconditioner_upd_interval=3,
                                                            curvature_upd_interval=2, ema_decay=0.1))
    assert [gm.do_update_preconditioner(s) for s in range(6)] == [True, False, False, True, False, False]
    assert [gm.do_update_curvature(s) for s in range(4)] == [True, False, True, False]
    assert gm.state_dict() == {'step': 0, 'curvature': {}}
    gm.load_state_dict({'step': 5})
    assert gm.state['step'] == 5
    gm2 = KfacGradientMaker(get_mlp(), PreconditioningConfig(data_size=1, num_total_steps=4,
                                                             preconditioner_upd_ratio=0.5))
    with pytest.warns(UserWarning):
        assert gm2.do_update_preconditioner(10) is False
    assert gm2.preconditioner_upd_schedule == [True, False, True, False] and gm2.curvature_upd_schedule is None
    assert [gm2.do_update_curvature(s) for s in range(4)] == [True, False, True, False]      # follows the preconditioner
    with pytest.warns(UserWarning):                      # a known horizon overrides the interval
        gm3 = KfacGradientMaker(get_mlp(), PreconditioningConfig(data_size=1, num_total_steps=4, ema_decay=0.1,
                                                                 preconditioner_upd_interval=2, curvature_upd_ratio=1.,
                                                                 preconditioner_upd_ratio=0.5))
    assert gm3.curvature_upd_schedule == [True] * 4 and gm3.do_update_curvature(1) and not gm3.do_update_preconditioner(1)
    gm4 = KfacGradientMaker(get_mlp(), PreconditioningConfig(data_size=1, preconditioner_upd_interval=4,
                                                             preconditioner_warmup_steps=3))
    assert [gm4.do_update_preconditioner(s) for s in range(9)] == [True] * 4 + [False] * 3 + [True, False]


def test_update_schedules_are_assignable_like_the_reference_attributes():
    """asdl/precondition/prec_grad_maker.py:85-99, 174-195: the schedules are plain attributes there; an assigned
    list decides step by step, None hands the decision back to the intervals."""
    model = get_mlp()
    gm = KfacGradientMaker(model, PreconditioningConfig(data_size=4, preconditioner_upd_interval=3))
    assert gm.preconditioner_upd_schedule is None and gm.curvature_upd_schedule is None
    assert [gm.do_update_preconditioner(s) for s in range(4)] == [True, False, False, True]
    gm.preconditioner_upd_schedule = [False, True, True, False]
    assert [gm.do_update_preconditioner(s) for s in range(4)] == [False, True, True, False]
    assert [gm.do_update_curvature(s) for s in range(4)] == [False, True, True, False]      # follows the preconditioner
    gm.curvature_upd_schedule = [True, True, False, False]
    assert [gm.do_update_curvature(s) for s in range(4)] == [True, True, False, False]
    gm.curvature_upd_schedule = None
    assert [gm.do_update_curvature(s) for s in range(4)] == [False, True, True, False]
    gm.preconditioner_upd_schedule = None
    assert [gm.do_update_preconditioner(s) for s in range(4)] == [True, False, False, True]


def test_module_selection_by_ignore_list_and_trainability():
    model = nn.Sequential(nn.Linear(3, 3), nn.ReLU(), nn.Linear(3, 3), nn.Sequential(nn.Linear(3, 2)), nn.Linear(2, 2))
    for p in model[4].parameters():
        p.requires_grad_(False)
    keys = lambda **kw: list(KfacGradientMaker(model, PreconditioningConfig(data_size=1, **kw)).module_dict.keys())
    assert keys() == ['0', '2', '3/0']                           # leaves with trainable parameters, '/' for '.'
    assert keys(ignore_modules=[model[0]]) == ['2', '3/0']
    assert keys(ignore_modules=['3.']) == ['0', '2']
    model_c = nn.Sequential(nn.Linear(3, 3), nn.Conv1d(3, 3, 1))
    with pytest.warns(UserWarning):
        assert list(KfacGradientMaker(model_c, PreconditioningConfig(data_size=1)).module_dict.keys()) == ['0']


def test_hooked_modules_follow_the_model_between_steps():
    """The list of hooked modules is kept between calls of no_centered_cov() and rebuilt when the module tree, a
    parameter object or a requires_grad flag has changed (the reference walks the modules at every call)."""
    from asdl_amd.core import no_centered_cov
    model = nn.Sequential(nn.Linear(3, 3), nn.ReLU(), nn.Linear(3, 3), nn.BatchNorm1d(3))

    def hooked(**kw):
        with no_centered_cov(model, ['kron'], **kw) as cxt:
            return [m for m in model.modules() if cxt.is_operation_registered(m) and m is not model]

    assert hooked(ignore_modules=[nn.BatchNorm1d]) == [model[0], model[2]]
    assert hooked(ignore_modules=[nn.BatchNorm1d]) == [model[0], model[2]]            # from the kept list
    assert len(model.__dict__['_asdl_amd_assignment_plans']) == 1
    for p in model[0].parameters():
        p.requires_grad_(False)
    assert hooked(ignore_modules=[nn.BatchNorm1d]) == [model[2]]                      # a frozen layer drops out
    model[0].weight.requires_grad_(True)
    assert hooked(ignore_modules=[nn.BatchNorm1d]) == [model[0], model[2]]
    new = nn.Linear(3, 3)
    model[2] = new                                                                    # a replaced module is picked up
    assert hooked(ignore_modules=[nn.BatchNorm1d]) == [model[0], new]
    model[0].weight = nn.Parameter(torch.zeros(3, 3), requires_grad=False)            # a replaced parameter too
    model[0].bias.requires_grad_(False)
    assert hooked(ignore_modules=[nn.BatchNorm1d]) == [new]
    assert hooked(ignore_modules=[new, nn.BatchNorm1d]) == []                         # other arguments, other list
    assert len(model.__dict__['_asdl_amd_assignment_plans']) == 2


def test_config_defaults_match_reference():
    c = PreconditioningConfig()
    assert (c.num_total_steps, c.preconditioner_upd_interval, c.preconditioner_warmup_steps) == (None, 1, 0)
    assert (c.curvature_upd_interval, c.curvature_upd_ratio, c.data_size, c.damping, c.ema_decay) == (None, None, -1, 1e-7, -1)
    assert c.ignore_modules is None and c.preconditioner_interval_type == 'constant'


def test_constructor_errors():
    from torch.nn.parallel import DistributedDataParallel
    model = nn.Sequential(nn.Embedding(4, 3), nn.Linear(3, 3), nn.BatchNorm1d(3))
    with pytest.raises(NotImplementedError, match='ignore_modules'):
        KfacGradientMaker(model, PreconditioningConfig(data_size=1))
    gm_bn = KfacGradientMaker(model, PreconditioningConfig(data_size=1, ignore_modules=[nn.Embedding]))
    assert gm_bn.shape_for[model[2]] == 'unit_wise' and gm_bn.shape_for[model[1]] == 'kron'
    with pytest.raises(NotImplementedError, match='unit-wise'):      # unit-wise blocks of a Linear layer are not built
        from asdl_amd.natural_gradient import NaturalGradientMaker
        NaturalGradientMaker(nn.Sequential(nn.Linear(3, 3)), PreconditioningConfig(data_size=1), fisher_shape='unit_wise')
    with pytest.raises(ValueError):
        KfacGradientMaker(get_mlp(), PreconditioningConfig(data_size=1, curvature_upd_ratio=0.5, num_total_steps=10))
    gm = KfacGradientMaker(get_mlp(), PreconditioningConfig())
    gm.setup_loss_call(F.cross_entropy, gm.setup_model_call(gm.model, torch.randn(2, 5)), torch.zeros(2, dtype=torch.long))
    with pytest.raises(ValueError, match='data_size'):
        gm.forward_and_backward()


# ------------------------------------------------------------------ K-FAC orchestration vs the reference's golden runs
@pytest.mark.parametrize('tag', sorted(GOLDEN_KFAC))
def test_kfac_host_logic_matches_reference_golden(tag, monkeypatch):
    cpu_backend.install(monkeypatch)
    factory, fisher_type, ema, damping, seed, ci, pi = GOLDEN_KFAC[tag]
    z = np.load(os.path.join(GOLDEN, f'kfac_{tag}.npz'))
    model = factory()
    model.load_state_dict({k[len('init/'):]: torch.from_numpy(z[k]) for k in z.files if k.startswith('init/')})
    bs = z['step0/x'].shape[0]
    config = PreconditioningConfig(data_size=bs, damping=damping, ema_decay=ema, curvature_upd_interval=ci,
                                   preconditioner_upd_interval=pi)
    gm = KfacGradientMaker(model, config, fisher_type=fisher_type, seed=seed, swift=tag.startswith('swift_'))
    opt = torch.optim.SGD(model.parameters(), lr=0.05)
    n_steps = len({k.split('/')[0] for k in z.files if k.startswith('step')})
    for step in range(n_steps):
        opt.zero_grad(set_to_none=True)
        x, t = torch.from_numpy(z[f'step{step}/x']), torch.from_numpy(z[f'step{step}/t'])
        dummy_y = gm.setup_model_call(model, x)
        gm.setup_loss_call(F.cross_entropy, dummy_y, t)
        y, loss = gm.forward_and_backward()
        torch.testing.assert_close(loss, torch.from_numpy(z[f'step{step}/loss']), rtol=1e-5, atol=1e-6)
        for name, p in model.named_parameters():
            assert grad_close(p.grad, torch.from_numpy(z[f'step{step}/grad/{name}']), 2e-4), (tag, step, name)
        for key in z.files:
            if key.startswith(f'step{step}/kron/'):
                _, _, mname, which = key.split('/')
                got = getattr(model.get_submodule(mname).fisher.kron, which)
                assert got is not None, key
                assert relerr(got, torch.from_numpy(z[key])) < 2e-4, key
            if key.startswith(f'step{step}/unit/'):
                _, _, mname, which = key.split('/')
                got = getattr(model.get_submodule(mname).fisher.unit, which)
                assert got is not None, key
                assert relerr(got, torch.from_numpy(z[key])) < 2e-4, key
        for name, m in model.named_modules():
            if isinstance(m, (nn.BatchNorm1d, nn.BatchNorm2d, nn.LayerNorm)) and ema == -1:
                assert m.fisher.unit.data is None and m.fisher.unit.has_inv
            if isinstance(m, (nn.Linear, nn.Conv2d)) and ema == -1:
                assert m.fisher.kron.A is None and m.fisher.kron.B is None    # only inverses are kept
        opt.step()
    assert gm.state_dict()['step'] == n_steps


@pytest.mark.parametrize('form', ['deep', 'plan', 'per module'])
def test_modules_that_share_a_gradient_are_preconditioned_one_after_the_other(form, monkeypatch):
    """Tied parameters: B2 (B1 G A1) A2 in the order of the modules.  The stand-ins for the launches that take many modules at
    once accept everything except what those launches cannot do, the same gradient twice."""
    import asdl_amd.natural_gradient as ng
    from asdl_amd import kernels
    from oracle import cpu_ref
    cpu_backend.install(monkeypatch)
    taken = []

    def distinct(addresses):
        assert len(set(addresses)) == len(addresses), 'one launch, the same gradient twice'
        taken.extend(addresses)

    def deep(items, units, grad_scale, device, fail=()):
        distinct([p for i in range(0, len(items), 6) for p in items[i + 2:i + 4] if p] + [p for i in range(0, len(units), 4) for p in units[i + 1:i + 3]])
        return False

    class Plan:
        def __init__(self, items, grad_scale=1.0, unit_items=()):
            distinct([g.data_ptr() for it in items for g in it[2:4] if g is not None] + [g.data_ptr() for it in unit_items for g in it[1:3]])
            self.items, self.grad_scale = items, grad_scale

        def launch(self):
            for B_inv, A_inv, g, b in self.items:
                cpu_backend.kron_precond(B_inv, A_inv, g, b, self.grad_scale)

    monkeypatch.setattr(ng, 'GROUPED_PRECONDITION', form != 'per module')
    monkeypatch.setattr(kernels, 'kron_precond_deep', deep)
    monkeypatch.setattr(kernels, 'kron_precond_groupable', lambda *a: True)
    monkeypatch.setattr(kernels, 'KronPrecondPlan', Plan)
    if form == 'deep':
        monkeypatch.setattr(ng, '_dense_on_gpu', lambda t, n: t is not None and t.numel() == n)
    torch.manual_seed(5)
    model = get_tied_mlp()
    reference = copy.deepcopy(model)
    x, t = torch.randn(16, 10), torch.randint(5, (16,))
    gm = KfacGradientMaker(model, PreconditioningConfig(data_size=16, damping=1e-2), fisher_type=FISHER_EMP, grad_scale=0.5)
    gm.setup_loss_call(F.cross_entropy, gm.setup_model_call(model, x), t)
    gm.forward_and_backward()
    assert bool(taken) == (form != 'per module')
    orc = cpu_ref.KfacOracle(reference, data_size=16, damping=1e-2, fisher_type='fisher_emp', unit_wise_norm=True, grad_scale=0.5)
    orc.forward_and_backward(x, t)
    for (name, p), q in zip(model.named_parameters(), reference.parameters()):
        assert grad_close(p.grad, q.grad, 2e-4), name


def _resume_run(monkeypatch, ema, ci, pi, fisher_type, n_steps=4, stop=2):
    """Gradients of an uninterrupted run and of one that is saved after ``stop`` steps and continued by a fresh
    maker on a fresh copy of the model."""
    cpu_backend.install(monkeypatch)
    torch.manual_seed(3)
    data = [(torch.randn(8, 5), torch.randint(4, (8,))) for _ in range(n_steps)]
    init = get_mlp().state_dict()

    def make():
        model = get_mlp()
        model.load_state_dict(init)
        config = PreconditioningConfig(data_size=8, damping=1e-2, ema_decay=ema, curvature_upd_interval=ci,
                                       preconditioner_upd_interval=pi)
        return model, KfacGradientMaker(model, config, fisher_type=fisher_type, seed=1), \
            torch.optim.SGD(model.parameters(), lr=0.05)

    def step(model, gm, opt, x, t):
        opt.zero_grad(set_to_none=True)
        gm.setup_loss_call(F.cross_entropy, gm.setup_model_call(model, x), t)
        gm.forward_and_backward()
        grads = [p.grad.clone() for p in model.parameters()]
        opt.step()
        return grads

    model, gm, opt = make()
    straight = [step(model, gm, opt, x, t) for x, t in data]
    model, gm, opt = make()
    resumed = [step(model, gm, opt, x, t) for x, t in data[:stop]]
    saved = gm.state_dict()
    weights = {k: v.clone() for k, v in model.state_dict().items()}
    for m in model.modules():                   # poison the live state: the clone in `saved` must not alias it
        fisher = getattr(m, 'fisher', None)
        if fisher is not None and fisher.has_kron:
            for attr in ('A', 'B', 'A_inv', 'B_inv'):
                if getattr(fisher.kron, attr) is not None:
                    getattr(fisher.kron, attr).fill_(float('nan'))
    model, gm, opt = make()
    model.load_state_dict(weights)
    gm.load_state_dict(saved)
    assert gm.state['step'] == stop
    resumed += [step(model, gm, opt, x, t) for x, t in data[stop:]]
    return straight, resumed, saved


@pytest.mark.parametrize('ema,ci,pi,fisher_type', [(-1, 3, 3, FISHER_EMP), (0.3, 1, 3, FISHER_EMP), (0.5, 2, 2, FISHER_MC)])
def test_state_dict_carries_the_curvature_through_a_resume(ema, ci, pi, fisher_type, monkeypatch):
    """Stop after step 2 of 4 with update intervals that make steps 2 and 3 depend on curvature computed earlier
    (stale inverses without EMA; running-average factors with EMA): the continued run has to reproduce the
    uninterrupted one bit for bit."""
    straight, resumed, saved = _resume_run(monkeypatch, ema, ci, pi, fisher_type)
    entry = saved['curvature']['0']
    assert {'kron.A_inv', 'kron.B_inv'} <= set(entry)
    assert ('kron.A' in entry) == (ema != -1)
    for a, b in zip(straight, resumed):
        for ga, gb in zip(a, b):
            assert torch.equal(ga, gb)


def test_load_state_dict_accepts_the_reference_form_and_rejects_unknown_modules():
    gm = KfacGradientMaker(get_mlp(), PreconditioningConfig(data_size=1))
    gm.load_state_dict({'step': 7})
    assert gm.state_dict() == {'step': 7, 'curvature': {}}
    with pytest.raises(KeyError, match='nosuch'):
        gm.load_state_dict({'step': 1, 'curvature': {'nosuch': {'kron.A': torch.eye(2)}}})


@pytest.mark.parametrize('per_call', [True, False])
def test_module_called_twice_in_one_forward(per_call, monkeypatch):
    """A module that is called twice per forward pass (shared weights), without EMA.  Default (the reference,
    asdl/operations/operation.py:225-233, 265-279, pinned by the golden runs 'shared_*'): every backward call inverts
    the pair (A of the LAST forward call, B of its own output gradient) with the pi-damping of that pair, and the
    inverses are added.  With operations.PER_CALL_INVERSES = False the contributions are summed and inverted once,
    (A1 + A2 + lam I)^-1."""
    import oracle.cpu_ref as R
    from asdl_amd import operations
    cpu_backend.install(monkeypatch)
    monkeypatch.setattr(operations, 'PER_CALL_INVERSES', per_call)
    torch.manual_seed(5)

    class Twice(nn.Module):
        def __init__(self):
            super().__init__()
            self.lin = nn.Linear(6, 6)
            self.head = nn.Linear(6, 3)

        def forward(self, x):
            return self.head(torch.tanh(self.lin(torch.tanh(self.lin(x)))))

    model = Twice()
    x, t = torch.randn(10, 6), torch.randint(3, (10,))
    ins, gouts = [], []
    def capture(m, i, o):
        ins.append(i[0].detach())
        o.register_hook(lambda g: gouts.append(g.detach()))
    handle = model.lin.register_forward_hook(capture)
    gm = KfacGradientMaker(model, PreconditioningConfig(data_size=10, damping=1e-2), fisher_type=FISHER_EMP)
    for _ in range(2):        # the second step reuses the per-call scratch buffers
        ins.clear(), gouts.clear()
        model.zero_grad(set_to_none=True)
        gm.setup_loss_call(F.cross_entropy, gm.setup_model_call(model, x), t)
        gm.forward_and_backward()
        assert len(ins) == 2 and len(gouts) == 2
        if per_call:
            A = R.linear_cov_kron_A(ins[-1]) / 10
            pairs = [R.kron_update_inv(A, R.linear_cov_kron_B(g) / 10, 1e-2) for g in gouts]
            A_inv, B_inv = sum(p[0] for p in pairs), sum(p[1] for p in pairs)
        else:
            A = sum(R.linear_cov_kron_A(a) for a in ins) / 10
            B = sum(R.linear_cov_kron_B(g) for g in gouts) / 10
            A_inv, B_inv = R.kron_update_inv(A, B, 1e-2)
        assert relerr(model.lin.fisher.kron.A_inv, A_inv) < 1e-5
        assert relerr(model.lin.fisher.kron.B_inv, B_inv) < 1e-5
    handle.remove()


# ------------------------------------------------------------------ FisherMaker invariants (test/grad_maker/test_fisher.py)
@pytest.mark.parametrize('network', ['mlp', 'cnn'])
@pytest.mark.parametrize('fisher_type', [FISHER_EMP, FISHER_MC, FISHER_EXACT])
@pytest.mark.parametrize('loss_type', [LOSS_CROSS_ENTROPY, LOSS_MSE])
def test_fisher_maker_invariants(network, fisher_type, loss_type, monkeypatch):
    cpu_backend.install(monkeypatch)
    torch.manual_seed(0)
    model = get_mlp() if network == 'mlp' else get_cnn()
    bs = 4
    x = torch.randn(bs, 5) if network == 'mlp' else torch.randn(bs, 5, 4, 4)
    t = torch.randint(4, (bs,)) if loss_type == LOSS_CROSS_ENTROPY else torch.randn(bs, 4)
    loss_fn = F.cross_entropy if loss_type == LOSS_CROSS_ENTROPY else F.mse_loss
    fm = get_fisher_maker(model, FisherConfig(fisher_type=fisher_type, fisher_shapes=[SHAPE_KRON], data_size=1,
                                              loss_type=loss_type, seed=1))
    fm.setup_loss_call(loss_fn, fm.setup_model_call(model, x), t)
    mods = [m for m in model.modules() if isinstance(m, (nn.Linear, nn.Conv2d))]

    def snap():
        return [(m.fisher.kron.A.clone(), m.fisher.kron.B.clone()) for m in mods]

    fm.forward_and_backward()
    first = snap()
    for m, (A, B) in zip(mods, first):
        in_dim = m.in_features if isinstance(m, nn.Linear) else m.in_channels * 4
        out_dim = m.out_features if isinstance(m, nn.Linear) else m.out_channels
        assert A.shape == (in_dim, in_dim) and B.shape == (out_dim, out_dim)
        torch.testing.assert_close(A, A.T)
        torch.testing.assert_close(B, B.T)
    for k in [2, 3]:                                     # test_accumulate
        fm.forward_and_backward(accumulate=True)
        for (A, B), (A1, B1) in zip(snap(), first):
            torch.testing.assert_close(A, A1 * k)
            torch.testing.assert_close(B, B1 * k)
    fm.forward_and_backward(scale=0.1)                   # test_scale
    for (A, B), (A1, B1) in zip(snap(), first):
        torch.testing.assert_close(A, A1 * 0.1)
    fm.forward_and_backward(data_size=32)                # test_data_size
    for (A, B), (A1, B1) in zip(snap(), first):
        torch.testing.assert_close(B, B1 / 32)
    damping = 1.0                                        # test_inv
    fm.forward_and_backward(calc_inv=True, damping=damping)
    for m, (A, B) in zip(mods, first):
        kron = m.fisher.kron
        assert kron.A is None and kron.B is None and kron.A_inv is not None and kron.B_inv is not None
        pi = torch.sqrt((A.trace() / A.shape[0]) / (B.trace() / B.shape[0]))
        dA, dB = max(damping ** 0.5 * pi, 1e-7), max(damping ** 0.5 / pi, 1e-7)
        torch.testing.assert_close(torch.eye(A.shape[0]), (A + dA * torch.eye(A.shape[0])) @ kron.A_inv)
        torch.testing.assert_close(torch.eye(B.shape[0]), (B + dB * torch.eye(B.shape[0])) @ kron.B_inv)
    N, damping = 10, 10.0                                # test_inv_data_size
    fm.forward_and_backward(calc_inv=True, damping=damping * N * N)
    inv1 = [(m.fisher.kron.A_inv.clone(), m.fisher.kron.B_inv.clone()) for m in mods]
    fm.forward_and_backward(data_size=N, calc_inv=True, damping=damping)
    for m, (Ai, Bi) in zip(mods, inv1):
        torch.testing.assert_close(m.fisher.kron.A_inv, Ai * N)
        torch.testing.assert_close(m.fisher.kron.B_inv, Bi * N)


@pytest.mark.parametrize('fisher_type', [FISHER_MC, FISHER_EXACT])
def test_pruned_fisher_backward_equals_full_backward(fisher_type, monkeypatch):
    """The sampled / exact passes differentiate with respect to the hooked module outputs only; every hook must
    still fire and see the same gradients, also when the first trainable module is a BatchNorm whose output an
    in-place ReLU overwrites, and the loss gradient that follows must be untouched."""
    import asdl_amd.fisher as fisher_mod
    cpu_backend.install(monkeypatch)

    def run(pruned):
        monkeypatch.setattr(fisher_mod, 'PRUNED_FISHER_BACKWARD', pruned)
        torch.manual_seed(3)
        model = nn.Sequential(nn.BatchNorm2d(5), nn.ReLU(inplace=True), nn.Conv2d(5, 6, 3, padding=1, bias=False),
                              nn.BatchNorm2d(6), nn.ReLU(inplace=True), nn.Conv2d(6, 4, 2), nn.Flatten(),
                              nn.Linear(4 * 3 * 3, 4))
        x, t = torch.randn(6, 5, 4, 4), torch.randint(4, (6,))
        gm = KfacGradientMaker(model, PreconditioningConfig(data_size=6, damping=1e-2, ema_decay=0.5),
                               fisher_type=fisher_type, seed=11)
        gm.setup_loss_call(F.cross_entropy, gm.setup_model_call(model, x), t)
        gm.forward_and_backward()
        out = {}
        for name, m in model.named_modules():
            f = getattr(m, 'fisher', None)
            if f is None:
                continue
            if f.has_kron:
                out[name + '.A'], out[name + '.B'] = f.kron.A.clone(), f.kron.B.clone()
            if f.has_unit:
                out[name + '.unit'] = f.unit.data.clone()
        for name, p in model.named_parameters():
            out['grad.' + name] = p.grad.clone()
        return out

    full, pruned = run(False), run(True)
    assert full.keys() == pruned.keys() and any(k.endswith('.unit') for k in full)
    for key in full:
        assert torch.equal(full[key], pruned[key]), key


# ------------------------------------------------------------------ side streams of the inverses
class _FakeStream:
    def __init__(self, handle):
        self.cuda_stream = handle


def test_threads_do_not_interleave_their_launches_on_one_side_stream(monkeypatch):
    """The pool of side streams is the process's and a stream's launches share its workspace: while one thread enqueues its
    groups on a stream, no other one may.  More groups than streams, so that all threads meet on all of them."""
    import threading
    import time
    from asdl_amd import kernels, symmatrix
    pool = [_FakeStream(h) for h in (11, 12, 13)]
    monkeypatch.setattr(symmatrix, '_side_streams', lambda dev, n: pool)
    monkeypatch.setattr(kernels, 'order_streams', lambda *a: None)
    busy, overlaps, ran = {}, [], []

    def run_group(group):
        handle = kernels._stream_handle()
        if busy.setdefault(handle, threading.get_ident()) != threading.get_ident():
            overlaps.append(handle)
        time.sleep(0.002)
        busy.pop(handle, None)
        ran.append(group)

    threads = [threading.Thread(target=lambda i=i: [symmatrix._enqueue_beside(None, [(i, k, j) for j in range(5)], run_group) for k in range(4)])
               for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert len(ran) == len(set(ran)) == 4 * 4 * 5
    assert not overlaps


def test_workspace_belongs_to_the_stream_whose_launches_use_it(monkeypatch):
    """A workspace that is replaced by a larger one goes back to the stream it was allocated on.  If that was the caller's stream
    while a side stream's launches used it, the caller's next tensor would take the memory under those launches."""
    from asdl_amd import kernels
    current, allocated = ['main'], []

    @contextlib.contextmanager
    def stream(st):
        current.append(st)
        yield
        current.pop()

    empty = torch.empty
    monkeypatch.setattr(torch.cuda, 'stream', stream)
    monkeypatch.setattr(torch, 'empty', lambda *a, **k: allocated.append(current[-1]) or empty(*a, **k))
    monkeypatch.setattr(kernels, '_workspaces', {})
    side = _FakeStream(77)
    with kernels.launches_on(side):
        for nbytes in (1 << 20, 1 << 22):
            kernels.workspace(nbytes, torch.device('cpu', 0))
    assert allocated == [side, side] and len(kernels._workspaces) == 1
    kernels.release_workspaces()
    assert not kernels._workspaces


def test_tables_on_the_device_belong_to_the_stream_that_reads_them(monkeypatch):
    """A cached table is uploaded asynchronously: another stream's launches would not wait for it, and when a cache is cleared its
    memory goes back to the stream it was uploaded on.  So every stream has its own."""
    from asdl_amd import kernels
    uploads = []

    def upload(host, device):
        uploads.append(kernels._stream_handle(device))
        return host.clone()
    monkeypatch.setattr(kernels, '_upload', upload)
    monkeypatch.setattr(kernels, '_capturing', lambda device: False)
    monkeypatch.setattr(kernels, '_tables', {})
    dev = torch.device('cuda', 0)
    plan = object.__new__(kernels.CholGroupPlan)
    plan.host, plan._dev = torch.zeros(8, dtype=torch.uint8), {}
    made = {}
    for _ in range(2):
        for handle in (3, 4):
            with kernels.launches_on(_FakeStream(handle)):
                made.setdefault(handle, []).append((kernels.device_ints((1, 2), dev), kernels.device_table(((1, 2),), dev),
                                                    kernels.device_addresses((1, 2), dev), plan.on_device(dev)))
    assert sorted(uploads) == [3] * 4 + [4] * 4
    for first, second in made.values():
        assert all(a is b for a, b in zip(first, second))
    assert all(a is not b for a, b in zip(made[3][0], made[4][0]))


def test_tables_made_under_a_stream_capture(monkeypatch):
    """The upload of such a table is a node of the graph: it reads the staged host memory at every replay, which therefore stays, and
    eager launches must not find a table that no replay has filled.  A table that a captured launch finds stays as well."""
    from asdl_amd import kernels
    capturing = [False]
    monkeypatch.setattr(kernels, '_tables', {})
    monkeypatch.setattr(kernels, '_kept_for_graphs', {})
    monkeypatch.setattr(kernels, '_capturing', lambda device: capturing[0])
    monkeypatch.setattr(kernels, '_upload', lambda host, device: host.clone())
    dev = torch.device('cuda', 0)
    with kernels.launches_on(_FakeStream(3)):
        eager = kernels.device_ints((1, 2), dev)
        capturing[0] = True
        assert kernels.device_ints((1, 2), dev) is eager
        inside = kernels.device_ints((3, 4), dev)
        capturing[0] = False
        assert kernels.device_ints((3, 4), dev) is not inside
        monkeypatch.setattr(kernels, '_workspaces', {})
        monkeypatch.setattr(kernels, '_on_launch_stream', contextlib.nullcontext)
        capturing[0] = True
        scratch, _ = kernels.workspace(1 << 20, torch.device('cpu', 0))
        capturing[0] = False
        kernels.release_workspaces()
    for t in (eager, inside, scratch):
        assert kernels._kept_for_graphs[id(t)] is t


def test_inverses_dropped_unfinished_are_waited_for(monkeypatch):
    """A pass beside the inverses that raises drops them unread: what takes their memory next has to run behind them."""
    from asdl_amd import kernels, symmatrix
    ordered = []
    monkeypatch.setattr(kernels, 'order_streams', lambda before, after, device: ordered.append((before, after)))
    side = _FakeStream(5)
    side.device = torch.device('cpu')
    pending = symmatrix.PendingInverses([], torch.zeros(1, dtype=torch.int32), None, [side], False)
    assert ordered == []
    del pending
    assert ordered == [(5, None)]


# ------------------------------------------------------------------ inverses that fail
@pytest.mark.parametrize('ema', [-1, 0.5])
@pytest.mark.parametrize('fisher_type', [FISHER_MC, FISHER_EMP])
@pytest.mark.parametrize('after', [True, False])
@pytest.mark.parametrize('earlier', [False, True])
def test_failed_inverses_are_not_kept(earlier, after, fisher_type, ema, monkeypatch):
    """A factor that is not positive definite raises from forward_and_backward(); who catches that and goes on must not find the
    failed inverse where the next step would precondition with it, whether the module had one before or not."""
    import asdl_amd.natural_gradient as ng_mod
    from asdl_amd import kernels
    cpu_backend.install(monkeypatch)
    monkeypatch.setattr(ng_mod, 'FLAGS_AFTER_PRECONDITION', after)
    broken, plain = [False], kernels.kron_damping

    def damping(A_list, B_list, *args, **kwargs):
        lam, nonzero = plain(A_list, B_list, *args, **kwargs)
        if broken[0]:
            lam[1] *= -1e6              # the second module's pair
        return lam, nonzero
    monkeypatch.setattr(kernels, 'kron_damping', damping)
    torch.manual_seed(2)
    model = get_mlp()
    x, t = torch.randn(8, 5), torch.randint(4, (8,))
    gm = KfacGradientMaker(model, PreconditioningConfig(data_size=8, damping=1e-2, ema_decay=ema), fisher_type=fisher_type, seed=1)

    def step():
        model.zero_grad(set_to_none=True)
        gm.setup_loss_call(F.cross_entropy, gm.setup_model_call(model, x), t)
        gm.forward_and_backward()
    if earlier:
        step()
    broken[0] = True
    with pytest.raises(torch.linalg.LinAlgError):
        step()
    broken[0] = False
    fisher = getattr(model[2], 'fisher', None)
    assert fisher is None or (fisher.kron.A_inv is None and fisher.kron.B_inv is None)
    step()
    assert model[2].fisher.kron.has_inv and all(torch.isfinite(p.grad).all() for p in model.parameters())


def test_singular_unit_wise_blocks_leave_the_earlier_inverse(monkeypatch):
    from asdl_amd import kernels, symmatrix
    flags = torch.tensor([[1, 0x7fffffff], [1, 4], [0, 0x7fffffff]], dtype=torch.int32)
    new = [torch.full((5, 2, 2), float(i)) for i in range(3)]
    old = [torch.eye(2).repeat(5, 1, 1) for _ in range(3)]
    monkeypatch.setattr(kernels, 'unit_wise_inv_grouped', lambda blocks, dampings: (list(new), flags))
    monkeypatch.setattr(kernels, 'unit_wise_keep_grouped', lambda invs, previous, fl: None)
    units = [symmatrix.UnitWise(torch.ones(5, 2, 2), inv) for inv in old]
    late = symmatrix.batched_unit_update_inv(units, 1e-2, late=True)
    with pytest.raises(torch.linalg.LinAlgError, match='block 3'):
        late.check(when=None)
    assert units[0].inv is new[0] and units[1].inv is old[1] and units[2].inv is old[2]


def test_all_flags_are_read_before_the_first_error_is_raised():
    from asdl_amd.symmatrix import read_flags
    seen = []

    class Late:
        def __init__(self, name, error=None):
            self.name, self.error = name, error

        def check(self, when='x'):
            seen.append((self.name, when))
            if self.error is not None:
                raise self.error
    with pytest.raises(torch.linalg.LinAlgError, match='first'):
        read_flags([Late('a'), Late('b', torch.linalg.LinAlgError('first')), Late('c', RuntimeError('second'))], when=None)
    assert seen == [('a', None), ('b', None), ('c', None)]
