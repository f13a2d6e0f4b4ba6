"""PUMAS tables on either side of the number of rows at which the envelope's
kernel changes: an element's rows do not depend on the others of the call (but
for the first, whose search takes the model everywhere), so they are the same
bit for bit."""
import numpy as np
import pytest
import torch

from noa_amd import pumas
from noa_amd.physics import MUON_MASS

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cutoff", [0.05, 1e-6])
def test_rows_across_the_line(device, cutoff):
    Z = np.arange(1., 20.)
    A = np.where(Z == 1., 1.008, 2.1 * Z)
    K = torch.logspace(-3, 9, 146, dtype=torch.float64, device=device)  # 3 x 19 x 146 = 8322 rows
    table, _, env = pumas.dcs_table(Z, A, MUON_MASS, cutoff, K)
    some = [0, 3, 4, 11, 17, 18]
    table_s, _, env_s = pumas.dcs_table(Z[some], A[some], MUON_MASS, cutoff, K)  # 2628 rows
    for a, b in ((table, table_s), (env, env_s)):
        assert torch.equal(a[:, some].nan_to_num(nan=-7.0), b.nan_to_num(nan=-7.0))
