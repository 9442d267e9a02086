"""Which parameters THORN.step takes as they are and which go through its full checks and working
copies: every kind in one group steps as it does alone, and what was refused stays refused."""
import pytest
import torch

import thorn_amd.optim as OPT
from thorn_amd import THORN

DEV = 'cuda:0'


class DTensor(torch.Tensor):   # the checks go by the type's name
    pass


def _opt(p, orthogonalize=True, **kw):
    return THORN([{'orthogonalize': orthogonalize, 'params': [p], 'lr': 1e-3, **kw}])


def test_refusals():
    p = torch.nn.Parameter(torch.zeros(4, 6))
    p.grad = torch.zeros(4, 6)
    with pytest.raises(RuntimeError, match='device tensors'):
        _opt(p).step()
    p.grad = torch.zeros(4, 6).to_sparse(1)
    with pytest.raises(RuntimeError, match='dense gradient'):
        _opt(p).step()
    p.grad = torch.zeros(4, 6).as_subclass(DTensor)
    with pytest.raises(NotImplementedError, match='DTensor'):
        _opt(p).step()
    p = torch.nn.Parameter(torch.zeros(4, 6, dtype=torch.complex64))
    p.grad = torch.zeros_like(p)
    with pytest.raises(NotImplementedError, match='supports'):
        _opt(p).step()
    p = torch.nn.Parameter(torch.zeros(4, 6))
    p.grad = torch.zeros(4, 6)
    with pytest.raises((RuntimeError, NotImplementedError, AssertionError)):
        _opt(p, orthogonalize=False, decouple_md=True).step()


KINDS = {
    'fp32': lambda t: (t, t),
    'bf16': lambda t: (t.bfloat16(), t.bfloat16()),
    'fp16': lambda t: (t.half(), t.half()),
    'fp64': lambda t: (t.double(), t.double()),
    'strided': lambda t: (t.t().contiguous().t(), t),
    'strided gradient': lambda t: (t, t.t().contiguous().t()),
    'strided bf16 gradient': lambda t: (t.bfloat16(), t.bfloat16().t().contiguous().t()),
}


@pytest.mark.gpu
@pytest.mark.parametrize('orthogonalize', [True, False])
@pytest.mark.parametrize('momentum_align', [False, True], ids=['', 'magma'])
def test_a_mixed_group_steps_as_its_parameters_alone(orthogonalize, momentum_align):
    print(f'[gpu] mixed group, orthogonalize {orthogonalize}, Magma {momentum_align}', flush=True)
    gen = torch.Generator().manual_seed(5)
    data = [(torch.randn(24, 40, generator=gen) * 0.05, torch.randn(3, 24, 40, generator=gen) * 1e-3) for _ in KINDS]
    idle = torch.randn(8, 8, generator=gen)

    def make():
        out = []
        for kind, (t, _) in zip(KINDS.values(), data):
            out.append(torch.nn.Parameter(kind(t.to(DEV))[0]))
        return out

    def step(opt, ps, which, k):
        for i in which:
            ps[i].grad = list(KINDS.values())[i](data[i][1][k].to(DEV))[1]
        opt.step()

    kw = dict(orthogonalize=orthogonalize, lr=1e-2, weight_decay=0.1, momentum_align=momentum_align)
    every = range(len(KINDS))
    group, alone = make(), make()
    unused = torch.nn.Parameter(idle.to(DEV))
    opt = THORN([{'params': [unused] + group, **kw}])
    opts = [THORN([{'params': [p], **kw}]) for p in alone]
    for k in range(3):
        step(opt, group, every[1:] if k == 2 else every, k)   # (once without the first one's gradient)
        if not momentum_align:   # (a Magma mask is drawn from the parameter's own seed)
            for i in every[1:] if k == 2 else every:
                step(opts[i], alone, [i], k)
    opt.check_status()
    torch.cuda.synchronize()
    assert torch.equal(unused.cpu(), idle) and 'step' not in opt.state[unused]
    for name, i in zip(KINDS, every):
        p = group[i]
        assert opt.state[p]['step'] == (3 if i == 0 else 4), name
        assert p.grad is None and torch.isfinite(p).all(), name
        if not momentum_align:
            assert torch.equal(p, alone[i]), name
            assert torch.equal(opt.state[p]['moment'], opts[i].state[alone[i]]['moment']), name


def test_release_windows_with_clusters_take_two_streams():
    """Small-matrix launches side by side must leave an XCD's 32 CUs a place for the last member of a cluster:
    a launch holds at most 15 for one that is not complete."""
    small, thin, large = (torch.empty(s, device='meta') for s in ((256, 640), (3, 128, 4096), (300, 4099)))
    streams = lambda w, orthogonalize=True: {OPT._release_stream(i, w, orthogonalize) for i in range(12)}
    for w in ([small], [thin], [large, small], [thin, large, large]):
        assert 15 * len(streams(w)) < 32 and streams(w) == {0, 1}
    assert streams([large]) == streams([large, large]) == {0, 1, 2}
    assert streams([small, thin], False) == {0, 1, 2}   # an Adam group has no clusters
