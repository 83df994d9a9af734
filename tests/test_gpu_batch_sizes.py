"""A batch chooses its fit and chain kernels by the voxels that run at once; its
volumes equal their separate runs, which choose by their own, to the last bit."""
import numpy as np
import pytest

from test_gpu_chain_paths import repeat, volume

pytestmark = pytest.mark.gpu


# (volumes, model, K) of each volume, their voxels: fits with a row per voxel in the batch and a wave alone (more than
# 24,576 voxels at once), Rician chains with one row in the batch and two alone (more than 6,144; three fibres keep
# two); the others stay below the lines
# (200 volumes with 18 of b = 0: the queue's tile of 18 against tiles of 14 alone, in one row and in two)
@pytest.mark.parametrize("vols,nvox,opts", [
    ([(200, 2, 3, 18), (220, 1, 2, 18)], 2301, {}), ([(200, 3, 2, 18), (112, 2, 3, 17)], 33, dict(f0=1)),
    ([(33, 1, 1), (69, 1, 2), (100, 2, 1), (48, 2, 2)], 6501, {}),
    ([(69, 2, 2), (33, 2, 1)], 2001, dict(f0=1)),
    ([(120, 2, 2), (160, 1, 1)], 3501, dict(rician=1)),
    ([(200, 2, 3), (161, 2, 2), (120, 1, 1)], 2401, dict(rician=1)),
    ([(300, 2, 2), (300, 2, 1)], 1501, {}),
    ([(33, 1, 1), (69, 2, 2), (145, 2, 1), (33, 2, 2), (120, 1, 2)], 601, dict(rician=1))])
def test_batch_equals_separate_runs(fdt, vols, nvox, opts):
    run = dict(opts, nburn=0, njumps=20, sampleevery=10)
    q = fdt.Queue()
    try:
        given = []
        for j, (n, model, K, *b0) in enumerate(vols):
            acq, data, _ = volume(n, 500, model, b0=b0[0] if b0 else max(2, n // 16), seed=j + 1)
            given.append((acq, repeat(data, nvox), dict(run, nfibres=K, model=model)))
            q.enqueue(*acq, given[-1][1], vox_offset=j * nvox, **given[-1][2])
        for _ in range(2):  # issued, then replayed
            q.run()
        for j, (acq, data, o) in enumerate(given):
            got, want = q.outputs(j), fdt.run_xfibres(*acq, data, vox_offset=j * nvox, **o)
            for k in got:
                np.testing.assert_array_equal(got[k], want[k], err_msg=f"volume {j} {vols[j]}: {k}")
    finally:
        q.close()
