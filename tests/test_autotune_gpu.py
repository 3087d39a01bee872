"""The plan autotuner (pw_autotune, in place of FFTW_MEASURE planning):
after tuning, H*psi still agrees with the oracle (the layouts differ only
in rounding order); the choice goes to the text cache and a second context
of the same shape applies it without timing."""
import numpy as np
import pytest

import oracle as O
from pwdft_develop_amd import workload as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name,nb", [("si8_32", 16), ("rand16_48", 12)])
def test_autotune_keeps_parity_and_caches(name, nb, tmp_path):
    import torch
    from pwdft_develop_amd.ops import Context
    print(f"case: autotune {name} nb={nb}", flush=True)
    prob = W.WORKLOADS[name](nb=nb).build()
    ref = O.Hamiltonian(prob).apply_h(prob.psi)
    cache = str(tmp_path / "tune.txt")
    for dt, tol in ((torch.complex128, 1e-11), (torch.complex64, 2e-5)):
        ctx = Context(prob)
        s1 = ctx.autotune(nb, dt, cache)
        assert "slab" in s1 and "cached" not in s1
        got = ctx.apply_h(ctx.to_device(prob.psi, dt)).cpu().numpy()
        assert np.abs(got - ref).max() < tol * np.abs(ref).max()
        ctx.close()
        ctx2 = Context(prob)
        s2 = ctx2.autotune(nb, dt, cache)
        assert "(cached)" in s2
        # the same slab choice and tiling come back from the file
        assert s2.split(" (")[0] == s1.split(" (")[0]
        got2 = ctx2.apply_h(ctx2.to_device(prob.psi, dt)).cpu().numpy()
        assert np.array_equal(got2, got)
        ctx2.close()
    lines = open(cache).read().splitlines()
    assert len(lines) == 4 and all("|" + f"{prob.grid[0]}x" in l for l in lines)


@pytest.mark.parametrize("value", ["reg 1 0", "reg 1 8 p", "lds 0 4 256"])
def test_slab_lines_of_other_choices_are_not_read(value, tmp_path):
    """A "slab" line, written by a tuner that knew no matrix-core kernel, does
    not keep a context from it: the slab is timed anew."""
    import torch
    from pwdft_develop_amd.ops import Context
    print(f"case: old cache line {value}", flush=True)
    prob = W.si8_32(nb=8).build()
    cache = tmp_path / "tune.txt"
    ctx = Context(prob)
    ctx.autotune(8, torch.complex64, str(cache))
    key, stage = cache.read_text().split()[0].rsplit("|", 1)
    cache.write_text(f"{key}|slab {value}\n")
    assert stage == "xy" and "(cached)" not in ctx.autotune(8, torch.complex64, str(cache))
    ctx.close()
