"""Batches whose events come in any order, with groups of fewer events than
subsets, images that are no multiple of a workgroup's voxels and arrays that
are not 16-byte aligned: equal to the reconstructions run one after another."""
import pytest
import torch

from tests import helpers as H

pytestmark = pytest.mark.gpu


def _recon(cuda, shape, n, seed, aligned):
    from srf_amd import preprocess, synth
    from srf_amd.data import Image, split_from_groups
    from srf_amd.scanner import CylindricalScanner
    sc = CylindricalScanner()
    size = (384.0, 384.0, 216.0)
    ev, _ = synth.tof_events(60_000, synth.c2_phantom(seed=3, scanner=sc), seed=seed, scanner=sc)
    groups = preprocess.recon_process(ev.to(cuda), sc.tof_res_ps)
    g = torch.Generator(device=cuda).manual_seed(seed)
    for a, k in zip("xyz", n):
        soa = groups[a]
        pick = torch.randperm(soa.shape[1], device=cuda, generator=g)[:k]
        groups[a] = soa[:, pick].contiguous()
    nv = shape[0] * shape[1] * shape[2]

    def array(lo):
        buf = torch.rand(nv + 4, device=cuda, generator=g) + lo
        o = 0 if aligned else 1
        return buf[o:o + nv].view(shape)

    return {"image": Image(array(0.5), (0, 0, 0), size), "emap": Image(array(0.5), (0, 0, 0), size),
            "data": split_from_groups(groups)}, sc


@pytest.mark.parametrize("schedule", [(4, 64), (1, 64), (16, 256)])
@pytest.mark.parametrize("kw", [9.0, 20.0, 36.0])
def test_unordered_batch(cuda, kw, schedule):
    """The same sums in another order: 1e-5, as every projector op."""
    from srf_amd import physics
    from srf_amd.batch import BatchedOSEM, serial_iterate
    from srf_amd.data import Image
    K = 3
    specs = [((41, 37, 29), (700, 2, 900), False), ((32, 32, 16), (5000, 4999, 0), True),
             ((16, 64, 4), (1, 64, 257), True)]
    recons = []
    for i, (shape, n, al) in enumerate(specs):
        r, sc = _recon(cuda, shape, n, 40 + i, al)
        recons.append(r)
    tb, ts2 = sc.tof_info()
    model = physics.SplitLoRsModel(kw, False, tof_sigma2=ts2, tof_bin=tb)
    b = [dict(r, image=Image(r["image"].data.clone(), (0, 0, 0), r["image"].size))
         for r in recons]
    bat = BatchedOSEM(recons, model, K)
    bat.set_schedule(*schedule)
    for rep in range(2):
        bat.iterate(1)
        serial_iterate(b, model, nb_subsets=K, nb_iterations=1)
        torch.cuda.synchronize()
        for ra, rb in zip(recons, b):
            e = H.rel_l2(ra["image"].data.cpu().numpy(), rb["image"].data.cpu().numpy())
            assert e <= 1e-5, (rep, e)
    bat.close()
