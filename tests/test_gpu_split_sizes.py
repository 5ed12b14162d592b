"""The split-precision step where its Legendre kernels stream their tables in
chunks (l_max > 255 or more than 384 theta rows): theta and l tiles that do not
fill a block, single levels, level groups of 16 with a remainder, m = 0 mod minc.
Every output within 1e-6 relative L2 of the FP64 form, the split form's bound."""
import pytest

from conftest import rel_l2
from magic_amd import sht
from nl_reference import make_inputs, radial
from test_gpu_split import SPLIT_TOL, _run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L,nt,nph,minc,nlev", [
    (256, 388, 768, 1, 1),    # 13 theta tiles, one level
    (300, 452, 320, 3, 9),    # second column tile of one level
    (341, 512, 1024, 1, 17),  # 16 theta tiles, a group of one level
    (40, 400, 96, 1, 16),     # one chunk, 13 theta tiles
    (15, 392, 48, 1, 5),      # fewer l than a chunk
])
def test_chunked_step_matches_fp64(L, nt, nph, minc, nlev):
    inputs = make_inputs(L, nlev, minc=minc)
    rad = radial(nlev)
    lcut = [L] * nlev
    lcut[nlev // 2] = L - 3
    p64 = sht.Plan(L, nt, nph, minc=minc, max_levels=nlev)
    ref = _run(p64, inputs, rad, lcut)
    p64.close()
    p16 = sht.Plan(L, nt, nph, minc=minc, precision=sht.PREC_SPLIT16, max_levels=nlev)
    outs = _run(p16, inputs, rad, lcut)
    p16.close()
    for k in range(10):
        assert rel_l2(outs[k], ref[k]) < SPLIT_TOL, sht.NL_OUTPUTS[k]
