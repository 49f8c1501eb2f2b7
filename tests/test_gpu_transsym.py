"""A TransSym table that leaves a site unmapped is refused: the tables built on
the device index by the map without looking at it again."""
import os

import pytest

pytestmark = pytest.mark.gpu


def test_unmapped_site_is_refused(tmp_path):
    import torch
    torch.zeros(1, device="cuda")
    import lattice
    import mvmc_hip
    info = lattice.write_workload("square8", str(tmp_path), seed=3, overrides=dict(L=4, nup=7, spgl=1, ntrans=2, walkers=2))
    path = os.path.join(str(tmp_path), "qptransidx.def")
    with open(path) as f:
        lines = f.readlines()
    assert len(lines[-1].split()) >= 3 and lines[-2].split()[0] == lines[-1].split()[0] == "1"
    lines[-1] = lines[-2]  # the last site of the second translation has no image
    with open(path, "w") as f:
        f.writelines(lines)
    with pytest.raises(mvmc_hip.BackendError, match="TransSym"):
        mvmc_hip.Ensemble(info["namelist"], info["initial"], walkers=2)
