"""The real-space path's matrix-core transforms at the edges of their tiles:
quarter planes of 7..63 rows, 5 to 32 columns (2 to 8 k-steps, one and two
tiles), unequal axes and refinements, fine axes equal to the coarse ones, odd
primes, one band and ragged groups, split projector sums, against the oracle.

Tolerance: psi passes three coarse and six fine chained sums, inner lengths at
most 32 or 63 each, 430 terms together, a rounding of one unit of the largest
partial sum in each: 512 eps of max |H psi|."""
import numpy as np
import pytest

import oracle as O
from pwdft_develop_amd import realspace as R

pytestmark = pytest.mark.gpu


def _problem(grid, fine, natom, nb):
    side = np.array(grid) * 0.42
    atoms = np.random.default_rng(natom).random((natom, 3)) * side
    species = [R.Species(0.9, (0.5, 0.6), (0.5, 0.7)) if i % 2 else R.Species(1.1, (0.4, 0.5), (0.45, 0.6))
               for i in range(natom)]
    return R.RealSpaceProblem("mm", tuple(grid), tuple(fine), np.diag(side), atoms, species, nb).build()


@pytest.mark.parametrize("grid,fine,natom,nb", [
    ((12, 14, 16), (24, 28, 32), 2, 1), ((16, 16, 16), (16, 16, 16), 3, 2), ((30, 32, 18), (60, 64, 36), 9, 5),
    ((62, 12, 16), (124, 24, 32), 4, 3), ((12, 62, 20), (24, 126, 40), 1, 6), ((16, 20, 62), (24, 34, 124), 0, 2),
    ((12, 16, 20), (24, 32, 20), 1, 6), ((12, 16, 20), (24, 16, 40), 1, 2),
    ((34, 34, 14), (68, 68, 28), 12, 9), ((64, 12, 12), (128, 24, 24), 3, 2),
    ((12, 16, 20), (12, 32, 40), 2, 3), ((64, 12, 14), (64, 24, 28), 2, 3), ((64, 12, 14), (64, 24, 14), 1, 2),
    ((12, 64, 14), (12, 64, 28), 2, 1), ((16, 64, 12), (32, 64, 24), 1, 2), ((14, 12, 64), (28, 24, 64), 2, 3)])
def test_matrix_core_transforms_against_oracle(grid, fine, natom, nb):
    import torch
    print(f"case: real-space transforms {grid} / {fine} natom={natom} nb={nb}", flush=True)
    if natom:
        p = _problem(grid, fine, natom, nb)
    else:
        p = _problem(grid, fine, 1, nb)
        p.npts, p.nproj = np.zeros(0, np.int32), np.zeros(0, np.int32)
        p.idx, p.val, p.wgt = np.zeros(0, np.int32), np.zeros(0), np.zeros(0)
    ref = O.rs_mult_spinor(p.grid, p.grid_fine, p.volume, p.ekin, p.vtot, p.npts, p.nproj, p.idx, p.val, p.wgt, p.psi)
    ctx = R.RealSpaceContext(p)
    x = torch.from_numpy(p.psi).cuda()
    got = ctx.mult_spinor(x).cpu().numpy()
    assert np.abs(got - ref).max() < 512 * 2.0 ** -53 * np.abs(ref).max()
    assert torch.equal(x.cpu(), torch.from_numpy(p.psi))
    # another potential and no projectors on the same handle, then back
    lib = R._lib.lib()
    R.check(lib.pw_rs_set_vtot(ctx.h, np.zeros_like(p.vtot)))
    bare = ctx.mult_spinor(x).cpu().numpy()
    zero = O.rs_mult_spinor(p.grid, p.grid_fine, p.volume, p.ekin, 0 * p.vtot, p.npts, p.nproj, p.idx, p.val, p.wgt,
                            p.psi)
    assert np.abs(bare - zero).max() < 512 * 2.0 ** -53 * np.abs(zero).max()
    R.check(lib.pw_rs_set_vtot(ctx.h, p.vtot))
    assert np.array_equal(ctx.mult_spinor(x).cpu().numpy(), got)
    ctx.close()


def test_refused_projectors_leave_the_potential():
    """Projector weights of more bytes than any card has (atoms without points,
    32 projectors each) are refused, and the handle then has no projectors:
    the whole of V psi, also on the old ones' points."""
    import torch
    p = _problem((12, 12, 12), (24, 24, 24), 2, 3)
    x = torch.from_numpy(p.psi).cuda()
    bare = R.RealSpaceContext(p, nonlocal_=False)
    want = bare.mult_spinor(x)
    ctx = R.RealSpaceContext(p, max_bands=1 << 20)
    print(f"case: refused projectors, chunk {ctx.info()['chunk']}", flush=True)
    assert not torch.equal(ctx.mult_spinor(x), want)
    natom = (1 << 42) // (8 * 32 * ctx.info()["chunk"])  # 4 TiB and more
    zero = np.zeros(natom, np.int32)
    with pytest.raises(RuntimeError, match="cannot allocate"):
        ctx.set_nonlocal(zero, zero + 32, np.zeros(0, np.int32), np.zeros(0), np.zeros(32 * natom))
    assert torch.equal(ctx.mult_spinor(x), want)
    ctx.set_nonlocal(p.npts, p.nproj, p.idx, p.val, p.wgt)
    ref = O.rs_mult_spinor(p.grid, p.grid_fine, p.volume, p.ekin, p.vtot, p.npts, p.nproj, p.idx, p.val, p.wgt, p.psi)
    assert np.abs(ctx.mult_spinor(x).cpu().numpy() - ref).max() < 512 * 2.0 ** -53 * np.abs(ref).max()
    ctx.close()
    bare.close()


def test_projector_weights_take_one_split_of_many_atoms():
    """48 GiB of projector weights at one value per projector and band (atoms
    too many to split their points) are accepted: several splits of them would
    exceed the card.  No atom has points here, so H psi is the bare one."""
    import torch
    p = _problem((12, 12, 12), (24, 24, 24), 2, 3)
    x = torch.from_numpy(p.psi).cuda()
    ctx = R.RealSpaceContext(p, max_bands=1 << 20, nonlocal_=False)
    want = ctx.mult_spinor(x)
    natom = (48 << 30) // (8 * 32 * ctx.info()["chunk"])
    print(f"case: many projectors, chunk {ctx.info()['chunk']} natom {natom}", flush=True)
    zero = np.zeros(natom, np.int32)
    ctx.set_nonlocal(zero, zero + 32, np.zeros(0, np.int32), np.zeros(0), np.zeros(32 * natom))
    assert torch.equal(ctx.mult_spinor(x), want)
    ctx.close()
