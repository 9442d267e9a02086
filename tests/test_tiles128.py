"""The two tile sizes of the Newton-Schulz launches (ns_phase_kernel's 256 x 256, ns_phase128_kernel's
128 x 128): the same sums in the same order, so the same steps bit for bit."""
import pytest
import torch

import thorn_amd.optim as OPT
from thorn_amd import THORN, _lib

DEV = 'cuda:0'


def _tile(shapes, flags=0):
    plan = _lib.OrthoPlan([r for r, _ in shapes], [c for _, c in shapes], [flags] * len(shapes))
    return _lib.load().thorn_ortho_tile(plan.handle)


def test_which_tiles_a_plan_takes():
    layer = lambda w: [(w, w), (w // 2, w), (w, w), (3 * w, w), (w, 3 * w)]
    for few in ([(257, 257)], [(300, 4099)], [(1500, 6000)], [(2048, 2048)], [(8192, 1024)], layer(320) * 20,
                layer(768), layer(1024)):
        assert _tile(few) == 128, few
    for many in ([(4096, 4096)], layer(768) * 20, layer(1024) * 8, layer(1024) * 20, [(8192, 8192), (16384, 1024)]):
        assert _tile(many) == 256, many
    assert _tile([(300, 520)], _lib.MAT_MD) == 256     # its sums of p^2 follow the tiles
    assert _tile([(300, 520)], _lib.MAT_TILES_256) == 256
    assert _tile([(4096, 4096)], _lib.MAT_TILES_128) == 128
    for md in (_lib.MAT_MD, _lib.MAT_MD_SCALAR):       # ... which the other kernel does not make
        with pytest.raises(RuntimeError, match='TILES_128'):
            _tile([(300, 520)], md | _lib.MAT_TILES_128)
        assert _tile([(64, 96)], md | _lib.MAT_TILES_128) == 128
    # a matrix of the small path has no such tiles and does not count
    assert _tile(layer(768) * 20 + [(64, 96)] * 500) == 256


# short sides around 128 and 256, long ones of one K tile more or less, tall (per row normalized), wide,
# square, widths of 8, 4, 2 and 1 whole elements; the last group gives each CU more than one tile
GROUPS = {
    'edges': [(257, 257), (256, 4096), (129, 8200), (8200, 130), (383, 640), (640, 385), (384, 384), (512, 513),
              (900, 1003), (1003, 900), (514, 1030), (260, 1036), (2, 300, 320)],
    'one': [(1024, 1024)],
    'two per CU': [(1024, 1024), (1024, 1100), (1100, 1024)] * 3,
}


@pytest.mark.gpu
@pytest.mark.parametrize('dtype', [torch.float32, torch.bfloat16], ids=['fp32', 'bf16'])
@pytest.mark.parametrize('group', GROUPS)
def test_tiles_give_the_same_steps(group, dtype, monkeypatch):
    print(f'[gpu] tiles of 128 and 256, {group}, {dtype}', flush=True)
    gen = torch.Generator().manual_seed(7)
    shapes = GROUPS[group]
    start = [(torch.randn(s, generator=gen) * 0.05).to(dtype) for s in shapes]
    steps = [[(torch.randn(s, generator=gen) * 1e-3).to(dtype) for s in shapes] for _ in range(3)]
    shapes_of = OPT._plan_shapes

    def run(flag):
        def forced(*args, **kw):
            out = list(shapes_of(*args, **kw))
            out[2] = [f | flag for f in out[2]]
            return tuple(out)
        monkeypatch.setattr(OPT, '_plan_shapes', forced)
        ps = [torch.nn.Parameter(t.to(DEV)) for t in start]
        opt = THORN([{'orthogonalize': True, 'params': ps, 'lr': 1e-2}])
        out = []
        for grads in steps:
            for p, g in zip(ps, grads):
                p.grad = g.to(DEV)
            opt.step()
            out.append([p.detach().clone() for p in ps])
        return out

    for k, (a, b) in enumerate(zip(run(_lib.MAT_TILES_128), run(_lib.MAT_TILES_256))):
        for s, x, y in zip(shapes, a, b):
            assert torch.isfinite(x).all(), (k, s)
            assert torch.equal(x, y), (k, s, (x - y).abs().max().item())
