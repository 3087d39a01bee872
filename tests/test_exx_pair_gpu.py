"""The register pair kernels of the exchange on the square planes that have
them, FP64 and FP32, against the oracle's three transforms a pair.

Tolerance: seven chained transforms of at most 7 radix passes, 4 eps each of
the largest value: 196 eps of max |V_x psi|.
"""
import numpy as np
import pytest

import oracle as O
from pwdft_develop_amd import workload as W

pytestmark = pytest.mark.gpu

SIDE = np.pi / np.sqrt(80.0)


@pytest.mark.parametrize("n,n3,fill,nb,nocc", [(24, 24, 0.99, 3, 2), (30, 10, 0.97, 2, 3), (32, 12, 0.999, 1, 1),
                                               (36, 10, 0.99, 2, 2), (40, 24, 0.95, 5, 3), (48, 10, 0.99, 2, 5),
                                               (60, 10, 0.99, 2, 2), (64, 10, 0.98, 2, 2), (72, 10, 0.99, 1, 3),
                                               (96, 10, 0.997, 2, 2)])
def test_pair_kernels_against_oracle(n, n3, fill, nb, nocc):
    import torch
    from pwdft_develop_amd.ops import Context
    sides = np.array([n, n, n3]) * SIDE * fill
    prob = W.Problem("pair", (n, n, n3), np.diag(sides), 10.0, sides[None, :] * [[0.3, 0.4, 0.6]], max(nb, nocc)).build()
    print(f"case: exchange pairs n={n} n3={n3} nb={nb} nocc={nocc}", flush=True)
    occ = np.linspace(1.0, 0.4, nocc)
    H = O.Hamiltonian(prob)
    H.set_exx(prob.ecut, 0.106, 0.25, prob.psi[:nocc], occ)
    ref = H.add_exx(prob.psi[:nb])
    ctx = Context(prob)
    ctx.set_exx(prob.ecut, 0.106, 0.25, ctx.to_device(prob.psi[:nocc]), occ)
    for dt, eps in ((torch.complex128, 2.0 ** -53), (torch.complex64, 2.0 ** -24)):
        got = ctx.add_exx(ctx.to_device(prob.psi[:nb], dt)).cpu().numpy()
        assert np.abs(got - ref).max() < 196 * eps * np.abs(ref).max()
    ctx.close()
