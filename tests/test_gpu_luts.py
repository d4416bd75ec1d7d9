"""Both forms of the Marschner table pass around their edges: tables smaller than
a workgroup, a partial last workgroup, and the sizes either side of the line
between the two.  Shared FP32 definitions: bit for bit with the oracle, NaN
texels at the same places."""
import numpy as np
import pytest

import barbu_amd as ba
from oracle import ftl_oracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("res", [2, 7, 9, 65, 362, 363, 500])
def test_forms_match_the_oracle(ctx, res):
    M, N = ba.marschner_luts(ctx, ba.marschner_params(eta=1.6, absorption=0.3, ar=-4.0, br=6.0), res)
    Mo, No = orc.marschner_luts(res, 1.6, 0.3, -4.0, 6.0)
    assert np.array_equal(M.view(np.uint32), Mo.view(np.uint32))
    nan = np.isnan(No)
    assert (np.isnan(N) == nan).all()
    assert np.array_equal(N[~nan].view(np.uint32), No[~nan].view(np.uint32))
