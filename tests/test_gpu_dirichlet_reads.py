"""One masked Dirichlet step without the cross term reads the mask of the four
neighbours only, so it takes well under the time of one with it, which reads
eight (4096 x 4096: 188 against 258 us; 254 with eight in both)."""
import pytest

import yolohtli_amd as Y
from timing import ratio
from yolohtli_amd import abi_types as T

pytestmark = pytest.mark.gpu


def test_no_diagonal_reads_without_the_cross_term(torch_cuda):
    torch = torch_cuda
    n = 4096
    a = [torch.from_numpy(x).cuda() for x in Y.initGates(n, n)]
    b = [torch.empty_like(x) for x in a]
    solid = torch.ones(n * n, dtype=torch.uint8, device="cuda")
    cross = dict(anisotropy=1, diff_par=0.0016, diff_per=0.0006, degrad=30.0)
    p, q = (T.grid_params(n, n, solidSwitch=1, neumannBC=0, **o) for o in ({}, cross))
    assert ratio(torch, lambda: Y.reactionDiffusion_wrapper(p, b, a, solid=solid),
                 lambda: Y.reactionDiffusion_wrapper(q, b, a, solid=solid), 10, 0.85) < 0.85
