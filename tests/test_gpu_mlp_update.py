"""The summing and Adam kernel of the weight network's training (k_mlp_update):
gradient and loss from 1 to 512 block partials (one block takes 64 samples),
and the packed operands it writes parameter by parameter."""
import numpy as np
import pytest

from microfc_amd import learned
from oracle import mlp as Q

from test_mlp_oracle import random_params, random_samples

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 64, 65, 1025, 32768, 40001])
def test_gradient_over_block_partials(gpu, n):
    torch = gpu
    P, S = random_params(21).astype(np.float32), random_samples(22, n).astype(np.float32)
    g, loss = learned.Mlp(P).gradient(torch.from_numpy(S).cuda())
    gr, lr = Q.gradient(P.astype(np.float64), S.astype(np.float64), bf16_points=True)
    # the bars of the 3001-sample gradient test: BF16 operands in another order
    assert loss == pytest.approx(lr, rel=1e-4)
    assert np.linalg.norm(g - gr) < 2e-2 * np.linalg.norm(gr)


def test_packed_operands_follow_the_parameters(gpu):
    torch = gpu
    S = torch.from_numpy(random_samples(23, 5000).astype(np.float32)).cuda()
    mlp = learned.Mlp(random_params(24).astype(np.float32))
    for _ in range(3):
        mlp.train_step(S, 1e-2)
    got, g, loss = mlp.infer(S).cpu().numpy(), *mlp.gradient(S)
    mlp.load(mlp.params())  # packs every operand from the parameters
    np.testing.assert_array_equal(mlp.infer(S).cpu().numpy(), got)
    g2, loss2 = mlp.gradient(S)
    np.testing.assert_array_equal(g2, g)
    assert loss2 == loss
