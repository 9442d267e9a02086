"""thorn::sym_addmm on operands that its product reads in place against the same operands copied
into its workspace: the same engine on the same values in the same order, so bit for bit."""
import ctypes
import math

import pytest
import torch

from thorn_amd import _lib

DEV = 'cuda:0'


def _needed(shape, a=(16, None), b=(16, None), c=None, c_mats=0):
    """Workspace of a call on tensors at the given addresses and strides (elements)."""
    nn, m, k = shape
    lib = _lib.load()
    i3 = lambda s: (ctypes.c_int64 * 3)(*s)
    sa = a[1] or (m * k, k, 1)
    sb = b[1] or (k * m, 1, k)
    return lib.thorn_sym_addmm_workspace_needed(a[0], i3(sa), b[0], i3(sb), c[0] if c else None,
                                                i3(c[1]) if c else None, c_mats, nn, m, k)


def test_which_operands_are_read_in_place():
    """The rule of the direct loads, from strides and addresses alone (no GPU)."""
    up = lambda v, q: -(-v // q) * q
    nn, m, k = 3, 40, 72
    copy = up(nn * m * up(k, 32) * 2, 256)
    assert _needed((nn, m, k)) == 0                                      # K-major A and B
    assert _needed((nn, m, k), b=(16, (k * m, m, 1))) == 0               # MN-major B
    assert _needed((nn, m, k), a=(16, (m * k, 1, m)), b=(16, (k * m, m, 1))) == 0   # MN-major both
    assert _needed((nn, m, k), a=(16, (m * k, 1, m))) == copy            # MN-major A, K-major B
    assert _needed((nn, m, k), a=(18, None)) == copy                     # address
    assert _needed((nn, m, k), a=(16, (m * k + 4, k, 1))) == copy        # matrix stride
    assert _needed((1, m, k), a=(16, (m * k + 4, k, 1))) == 0            # ... of a single product
    assert _needed((nn, m, k), a=(16, (m * 76, 76, 1))) == copy          # line stride
    assert _needed((nn, m, k), a=(16, (m * 80, 80, 1))) == 0
    assert _needed((nn, m, k), a=(16, (0, 2 * k, 2))) == copy            # no unit stride
    assert _needed((nn, m, 70)) == 2 * up(nn * m * 96 * 2, 256)          # lengths
    assert _needed((nn, 36, k), b=(16, (k * 40, 40, 1))) == up(nn * 36 * 96 * 2, 256)
    assert _needed((nn, m, k), b=(16, (k * m, 32, 1))) == copy           # MN-major lines overlap
    mat, row = (m * m, m, 1), (m * 48, 48, 1)
    assert _needed((nn, m, k), c=(32, mat), c_mats=nn) == 0
    assert _needed((nn, m, k), c=(32, (7, m, 1)), c_mats=1) == 0         # one C: no matrix stride
    assert _needed((nn, m, k), c=(32, row), c_mats=nn) == up(nn * m * m * 2, 256)
    assert _needed((nn, m, k), c=(34, mat), c_mats=nn) == up(nn * m * m * 2, 256)
    assert _needed((nn, m, 0)) == 2 * up(nn * m * 32 * 2, 256)           # nothing to read
    lib = _lib.load()
    assert lib.thorn_sym_addmm_workspace_bytes(nn, m, k, nn) == 2 * copy + up(nn * m * m * 2, 256)


def _off_by_one(t):
    """The same values at an address that is no multiple of 16 bytes: copied into the workspace."""
    buf = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)
    return torch.as_strided(buf, t.shape, torch.empty(t.shape).stride(), 1).copy_(t)


# m and k at the edges of a tile (256), of a K tile (32) and of a chunk (8)
SHAPES = [(1, 8, 8), (2, 248, 32), (2, 256, 40), (3, 264, 120), (1, 520, 128), (2, 512, 1000), (1, 776, 24),
          (2, 40, 4104)]


@pytest.mark.gpu
@pytest.mark.parametrize('shape', SHAPES, ids=lambda s: 'x'.join(map(str, s)))
def test_in_place_equals_copied(shape):
    import thorn_amd  # noqa: F401
    import thorn_amd.ops  # noqa: F401
    nn, m, k = shape
    print(f'[gpu] sym_addmm in place {shape}', flush=True)
    gen = torch.Generator().manual_seed(m + k)
    op = torch.ops.thorn.sym_addmm
    wide = torch.randn(nn, m, k + 16, generator=gen).half().to(DEV) / math.sqrt(k)
    x = wide[..., :k].contiguous()
    s = torch.randn(nn, m, m, generator=gen)
    s = ((s + s.mT) / math.sqrt(m)).half().to(DEV)
    xt = x.mT.contiguous()
    for name, a, b, c in (('gram', x, x.mT, None), ('strided rows', wide[..., :k], wide[..., :k].mT, s),
                          ('b by columns', x, xt, s), ('both by columns', xt.mT, xt, s[0]), ('poly', s, s, s),
                          ('a by columns', xt.mT, x.mT, None), ('one for all', x[:1].expand_as(x), x[0].mT.expand(nn, k, m), s)):
        got = op(a, b, c, 0.75, -1.5)
        want = op(_off_by_one(a), _off_by_one(b), None if c is None else _off_by_one(c), 0.75, -1.5)
        assert torch.equal(got, want), name
        assert torch.equal(got, got.mT), name
        exact = 0.75 * (a.double() @ b.double().contiguous()) + (0 if c is None else -1.5 * c.double())
        # one rounding to f16 (2^-11 of each value) of a sum in fp32
        err = (got.double() - exact).norm() / exact.norm()
        assert err <= 2.0 ** -11, (name, err)


@pytest.mark.gpu
def test_in_place_reads_nothing_behind_the_operand():
    """An operand's end, its rows' padding and what lies past k are NaN: none of it reaches a result."""
    import thorn_amd.ops  # noqa: F401
    print('[gpu] sym_addmm in place, NaN around the operands', flush=True)
    m, k = 296, 200
    gen = torch.Generator().manual_seed(5)
    v = torch.randn(m, k, generator=gen).half().to(DEV)
    buf = torch.full((m + 300, k + 24), float('nan'), dtype=torch.float16, device=DEV)
    x = buf[:m, :k]
    x.copy_(v)
    bufc = torch.full((k + 300, m + 8), float('nan'), dtype=torch.float16, device=DEV)
    xt = bufc[:k, :m]
    xt.copy_(v.mT)
    want = torch.ops.thorn.sym_addmm(v, v.mT.contiguous(), None, 1.0, 0.0)
    for a, b in ((x, x.mT), (x, xt), (xt.mT, xt)):
        assert torch.equal(torch.ops.thorn.sym_addmm(a, b, None, 1.0, 0.0), want)


def _call(lib, a, sa, b, sb, c, sc, c_mats, out, shape, beta, ws, nbytes, stream=None):
    i3 = lambda s: (ctypes.c_int64 * 3)(*s)
    return lib.thorn_sym_addmm(a, i3(sa), b, i3(sb), c, i3(sc) if c else None, c_mats, out, *shape, 1.0, beta, ws, nbytes,
                               stream)


def test_out_over_an_operand_needs_its_copy():
    """Operands that could be read in place, beside an out that shares memory with one of them: refused without
    the workspace for its copy (on the host, before anything is launched)."""
    lib = _lib.load()
    nn, m = 2, 256
    mat = (m * m, m, 1)
    size = 2 * nn * m * m
    a, b, c = (size * i for i in range(1, 4))
    for sc, c_mats, out in ((None, 0, a), (None, 0, a - 16), (None, 0, a + size - 16), (None, 0, b + size // 2), (mat, nn, b),
                            (mat, nn, c + size // 2),                     # a matrix off C
                            ((0, m, 1), 1, c),                            # one C for two products
                            ((2 * m * m, m, 1), nn, c)):                  # C of other strides
        rc = _call(lib, a, mat, b, mat, c if sc else None, sc, c_mats, out, (nn, m, m), 1.0, None, 0)
        assert rc != 0 and 'workspace' in lib.thorn_last_error().decode(), (sc, c_mats, out)


@pytest.mark.gpu
@pytest.mark.parametrize('shape', [(3, 512, 512), (2, 520, 40), (1, 264, 264), (2, 250, 250)],
                         ids=lambda s: 'x'.join(map(str, s)))
def test_out_over_an_operand(shape):
    nn, m, k = shape
    print(f'[gpu] sym_addmm, out over an operand, {shape}', flush=True)
    lib = _lib.load()
    gen = torch.Generator().manual_seed(m + k + 1)
    n_ab, n_out = nn * m * k, nn * m * m
    pool = torch.randn(4 * max(n_ab, n_out) + 4096, generator=gen).half().to(DEV)
    nbytes = lib.thorn_sym_addmm_workspace_bytes(nn, m, k, nn)
    ws = torch.empty(nbytes, dtype=torch.uint8, device=DEV)
    ab, mat = (m * k, k, 1), (m * m, m, 1)
    for name, at_a, at_c, at_out in (('a', 0, None, 0), ('inside a', 2048, None, 0), ('across b', 0, None, n_ab // 2 // 8 * 8),
                                     ('c', 0, n_ab, n_ab), ('c, shifted', 0, n_ab + 64, n_ab)):
        buf = pool.clone()
        a = buf[at_a:at_a + n_ab].view(nn, m, k)
        c = None if at_c is None else buf[at_c:at_c + n_out].view(nn, m, m)
        want = torch.ops.thorn.sym_addmm(a, a.mT, c, 1.0, -0.5)
        needed = nbytes if name != 'c' or m % 8 or k % 8 else 0   # C may be out itself
        rc = _call(lib, a.data_ptr(), ab, a.data_ptr(), (m * k, 1, k), c.data_ptr() if c is not None else None, mat,
                   0 if c is None else nn, buf.data_ptr() + 2 * at_out, shape, -0.5, ws.data_ptr() if needed else None,
                   needed, torch.cuda.current_stream().cuda_stream)
        assert rc == 0, (name, lib.thorn_last_error())
        assert torch.equal(buf[at_out:at_out + n_out].view(nn, m, m), want), name
