"""What an operator does with its operand and stream: arrays that are ready are passed through, every other
form is converted, and the work goes to torch's current stream."""

import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gf():
    import torch

    import goosefem_amd

    assert torch.cuda.is_available(), "GPU tests need a GPU"
    goosefem_amd.lib()
    return goosefem_amd


def test_operand_forms(gf):
    import torch

    a = np.random.default_rng(0).standard_normal((6, 4))
    d = torch.from_numpy(a).cuda()
    assert gf.to_device(d) is d and gf.to_device(d.float(), torch.float32).dtype == torch.float32
    wide = torch.zeros((6, 8), dtype=torch.float64, device="cuda")
    wide[:, ::2] = d
    c, conn = oracle.quad4_regular(2, 1)
    vec = gf.Vector(conn, oracle.dofs(6, 2))
    ref = oracle.Vector(conn, oracle.dofs(6, 2)).AsElement(np.ascontiguousarray(a[:, :2]))
    b = np.ascontiguousarray(a[:, :2])
    forms = (b, torch.from_numpy(b), torch.from_numpy(b).cuda(), d[:, :2], wide[:, 0:4:2],
             torch.from_numpy(np.asfortranarray(b)).cuda())
    for x in forms:
        assert np.array_equal(vec.AsElement(x).cpu().numpy(), ref)
    for x in (b.astype(np.float32), torch.from_numpy(b.astype(np.float32)).cuda()):
        want = oracle.Vector(conn, oracle.dofs(6, 2)).AsElement(b.astype(np.float32).astype(np.float64))
        assert np.array_equal(vec.AsElement(x).cpu().numpy(), want)
    ints = torch.arange(3, device="cuda")
    assert gf.to_device(ints).dtype == torch.int64


def test_work_goes_to_the_current_stream(gf):
    import torch

    assert (gf._stream().value or 0) == torch.cuda.current_stream().cuda_stream  # ctypes: None for a null pointer
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        assert gf._stream().value == s.cuda_stream
