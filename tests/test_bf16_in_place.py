"""bf16 parameters stepped in place against the same parameters stepped through fp32 working copies:
the same fp32 arithmetic on the same values with one rounding at the end, so bit for bit."""
import pytest
import torch

import thorn_amd.optim as OPT
from thorn_amd import THORN, _lib

DEV = 'cuda:0'


def test_bf16_plans_refuse_what_needs_fp32_state():
    plan = _lib.OrthoPlan([8, 16], [16, 8], [_lib.MAT_BF16, _lib.MAT_BF16 | _lib.MAT_PER_ROW_NORM])
    assert plan.workspace_bytes > 0
    for f in (_lib.MAT_MD, _lib.MAT_MD_SCALAR, _lib.MAT_MD | _lib.MAT_ADAM):
        with pytest.raises(RuntimeError):
            _lib.OrthoPlan([8], [16], [_lib.MAT_BF16 | f])


# the fused and separate small launches, edge tiles, rows of 8, 4, 2 and 1 whole elements, tall (per
# row normalized), wide, square, a batch of matrices, and sizes that take the prescaled first iterate
SHAPES = [(32, 5), (64, 96), (256, 640), (640, 256), (300, 520), (257, 258), (301, 1003), (3, 288, 320), (520, 300),
          (1024, 1024), (1100, 1020), (1000, 1052), (1024, 2048), (1536, 1024)]
VECS = [(1,), (7,), (4096,), (12289,), (3, 4100)]


@pytest.mark.gpu
@pytest.mark.parametrize('rate', [1, 2])
def test_in_place_equals_working_copies(rate, monkeypatch):
    print(f'[gpu] bf16 in place, update rate {rate}', flush=True)
    gen = torch.Generator().manual_seed(11)
    start = [(torch.randn(s, generator=gen) * 0.05).to(torch.bfloat16) for s in SHAPES + VECS]
    steps = []
    for k in range(4):   # the third step's gradients fall by 1e-4 (the first iterate is rebuilt), the fourth's rise
        scale = (1e-3, 1e-3, 1e-7, 1.0)[k]
        steps.append([(torch.randn(s, generator=gen) * scale).to(torch.bfloat16) for s in SHAPES + VECS])

    def run(copies):
        if copies:
            monkeypatch.setattr(OPT, '_needs_shadow', lambda p, group, state: p.dtype == torch.bfloat16)
        else:
            monkeypatch.undo()
        ps = [torch.nn.Parameter(t.to(DEV)) for t in start]
        n, k = len(SHAPES), len(SHAPES) + 2
        opt = THORN([{'orthogonalize': True, 'params': ps[:n], 'lr': 2e-2, 'betas': (0.1, 0.95)},
                     {'orthogonalize': False, 'params': ps[n:k], 'lr': 1e-2},
                     {'orthogonalize': False, 'params': ps[k:], 'lr': 1e-2, 'eps': 1e-8, 'rectify': True,
                      'weight_decay': 0.0}])
        opt._update_rate = rate
        out = []
        for grads in steps:
            for p, g in zip(ps, grads):
                p.grad = g.to(DEV)
            opt.step()
            out.append([p.detach().clone() for p in ps] +
                       [v.clone() for p in ps for v in opt.state[p].values() if torch.is_tensor(v)])
        assert bool(opt._shadows) == copies
        return out

    for k, (a, b) in enumerate(zip(run(False), run(True))):
        for i, (x, y) in enumerate(zip(a, b)):
            assert x.dtype == torch.bfloat16
            assert torch.equal(x, y), (k, i, tuple(x.shape), (x.float() - y.float()).abs().max().item())


# a resumed run: moments that are not zero and the default beta1, so that the moment's rounding to bf16
# takes something off in nearly every element (of 0.9 m + g one in thirty falls on the middle of two bf16
# values). 'large': the first iterate made by a launch of its own, on the first step and on the third, whose
# gradients jump; enough elements for one changed unit of u to change an iterate. 'small': the fused launch
# from the second step on, with u kept in registers and, for the widest, read again
RESUMED = {'large': [(1024, 3072), (3072, 1024), (1000, 3072), (1024, 3070), (64, 96)],
           'small': [(16, 3072), (200, 4001), (640, 256), (3072, 48), (96, 64), (128, 128), (3000, 129), (255, 255),
                     (16, 65000)]}


@pytest.mark.gpu
@pytest.mark.parametrize('group,tiles', [('large', 128), ('large', 256), ('small', 0)])
def test_first_iterate_takes_the_unrounded_moment(group, tiles, monkeypatch):
    print(f'[gpu] bf16 in place, resumed, {group}, tiles of {tiles}', flush=True)
    gen = torch.Generator().manual_seed(13)
    shapes = RESUMED[group]
    shapes_of = OPT._plan_shapes

    def forced(*args, **kw):   # (both sizes of tiles have a kernel of their own for the last update)
        rows, cols, flags, *rest = shapes_of(*args, **kw)
        flag = {128: _lib.MAT_TILES_128, 256: _lib.MAT_TILES_256, 0: 0}[tiles]
        return (rows, cols, [f | flag for f in flags], *rest)
    start, moments = ([(torch.randn(s, generator=gen) * f).to(torch.bfloat16) for s in shapes] for f in (0.02, 2e-3))
    steps = [[(torch.randn(s, generator=gen) * f).to(torch.bfloat16) for s in shapes] for f in (1e-3, 1e-3, 0.1)]

    def run(copies):
        if copies:
            monkeypatch.setattr(OPT, '_needs_shadow', lambda p, group, state: p.dtype == torch.bfloat16)
        else:
            monkeypatch.undo()
        monkeypatch.setattr(OPT, '_plan_shapes', forced)
        ps = [torch.nn.Parameter(t.to(DEV)) for t in start]
        opt = THORN([{'orthogonalize': True, 'params': ps, 'lr': 2e-2, 'betas': (0.9, 0.95)}])
        for p, m in zip(ps, moments):
            opt.state[p].update(step=10, moment=m.to(DEV))
        out = []
        for grads in steps:
            for p, g in zip(ps, grads):
                p.grad = g.to(DEV)
            opt.step()
            out.append([p.detach().clone() for p in ps] + [opt.state[p]['moment'].clone() for p in ps])
        assert bool(opt._shadows) == copies
        opt.check_status()
        return out

    for k, (a, b) in enumerate(zip(run(False), run(True))):
        for s, x, y in zip(shapes * 2, a, b):
            assert torch.equal(x, y), (k, s, (x != y).sum().item())


@pytest.mark.gpu
def test_chains_in_place():
    """A bf16 group that steps as two chains, each with its prologue on a stream of its own, against the same group
    as one plan and as chains of working copies: a resumed run whose gradients jump in the third step (the first
    iterate is made again from the moment before the step)."""
    print('[gpu] bf16 in place, two chains', flush=True)
    gen = torch.Generator().manual_seed(14)
    shapes = [(384, 640), (640, 384), (512, 512), (1024, 384), (96, 640)] * 5 + [(3, 384, 512)]
    start, moments = ([(torch.randn(s, generator=gen) * f).to(torch.bfloat16) for s in shapes] for f in (0.02, 2e-3))
    steps = [[(torch.randn(s, generator=gen) * f).to(torch.bfloat16) for s in shapes] for f in (1e-3, 1e-3, 0.1)]

    def run(chains, copies):
        with pytest.MonkeyPatch.context() as mp:
            mp.setattr(OPT, 'CHAIN_MIN_MATRICES', 16 if chains else 1 << 30)
            mp.setattr(OPT, 'CHAIN_MIN_COST', 0)
            if copies:
                mp.setattr(OPT, '_needs_shadow', lambda p, group, state: True)
            ps = [torch.nn.Parameter(t.to(DEV)) for t in start]
            opt = THORN([{'orthogonalize': True, 'params': ps, 'lr': 2e-2, 'betas': (0.9, 0.95)}])
            for p, m in zip(ps, moments):
                opt.state[p].update(step=10, moment=m.to(DEV))
            out = []
            for grads in steps:
                for p, g in zip(ps, grads):
                    p.grad = g.to(DEV)
                opt.step()
                out.append([p.detach().clone() for p in ps] + [opt.state[p]['moment'].clone() for p in ps])
            assert next(iter(opt._runners.values())).chained == chains and bool(opt._shadows) == copies
            opt.check_status()
            return out

    chained = run(True, False)
    for other in (run(False, False), run(True, True)):
        for k, (a, b) in enumerate(zip(chained, other)):
            for s, x, y in zip(shapes * 2, a, b):
                assert torch.equal(x, y), (k, s, (x != y).sum().item())


@pytest.mark.gpu
def test_unaligned_bf16_tensors():
    """Parameters, gradients and moments at odd addresses take the element-wise loads: the sums over
    a tile run in another order, so the update may differ in its last places."""
    print('[gpu] bf16 in place, unaligned', flush=True)
    gen = torch.Generator().manual_seed(12)
    shapes = [(64, 96), (300, 520), (1024, 1032), (4100,)]

    def odd(t):
        buf = torch.empty(t.numel() + 1, dtype=t.dtype, device=DEV)
        return buf[1:].view(t.shape).copy_(t)

    start = [(torch.randn(s, generator=gen) * 0.05).to(torch.bfloat16) for s in shapes]
    grads = [[(torch.randn(s, generator=gen) * 1e-3).to(torch.bfloat16) for s in shapes] for _ in range(2)]
    ends = []
    for place in (lambda t: t.to(DEV), odd):
        ps = [torch.nn.Parameter(place(t)) for t in start]
        opt = THORN([{'orthogonalize': True, 'params': ps[:3], 'lr': 2e-2},
                     {'orthogonalize': False, 'params': ps[3:], 'lr': 1e-2}])
        for step in grads:
            for p, g in zip(ps, step):
                p.grad = place(g)
            opt.step()
        assert not opt._shadows
        ends.append([p.detach().float() for p in ps] + [opt.state[p]['moment'].float() for p in ps])
    n = len(shapes)
    for i, (x, y) in enumerate(zip(*ends)):
        # a bf16 value next to the middle of two goes either way: 2^-8 of it, in few values
        assert ((x - y).abs() <= 2.0 ** -7 * x.abs() + 1e-12).all(), i
        assert (x != y).float().mean() <= (0.02 if i < n else 0.0), i
