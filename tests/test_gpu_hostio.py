"""Calls on host arrays: what fits the context's pinned memory (4 MiB a call)
goes through it, what does not is copied directly; same results."""
import numpy as np
import pytest

import oracle
from kernel_check import device_events
from mcvslam_amd import Context, Matcher, ORB, synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def own_ctx(gpu_ctx):
    ctx = Context(0)
    yield ctx
    ctx.close()


def test_parts_to_host_sizes_and_alignments(own_ctx):
    """More ranges than one launch copies, of sizes around 16 bytes and one
    workgroup's share, at every alignment, one larger than the pinned memory,
    one empty."""
    import torch
    src = torch.randint(0, 256, (6 << 20,), dtype=torch.uint8, device="cuda")
    ref = src.cpu().numpy()
    torch.cuda.synchronize()
    parts = [(1, 1), (2, 15), (3, 16), (0, 17), (5, 16384), (6, 16385), (7, 70000), (8, 0), (9, 5 << 20), (11, 4095),
             (13, 31)]
    for group in (parts, parts[:8], parts[8:]):
        outs = own_ctx.to_host_all([(src.data_ptr() + o, np.uint8, (n,)) for o, n in group])
        for (o, n), a in zip(group, outs):
            np.testing.assert_array_equal(a, ref[o:o + n], err_msg=str((o, n)))


@pytest.mark.parametrize("nq,nt", [(1, 1), (3, 140000), (140000, 3)])
def test_match_sizes(own_ctx, nq, nt):
    rng = np.random.default_rng(nq + nt)
    q, t = (rng.integers(0, 256, (n, 32), dtype=np.uint8) for n in (nq, nt))
    rows = Matcher.KnnMatch(q, t, ctx=own_ctx)
    np.testing.assert_array_equal(rows.rows, oracle.knn2(q, t))


def test_large_image(own_ctx):
    """2400 x 1800: larger than the pinned memory."""
    img = synth.blob_image(5, 2400, 1800)
    kps, desc = ORB(2000, 1.2, 8, 20, 7, ctx=own_ctx).extract(img)
    rk, rd = oracle.orb_extract(img, 2000, 1.2, 8, 20, 7)
    for f in ("x", "y", "size", "angle", "response", "octave"):
        np.testing.assert_array_equal(kps[f], rk[f], err_msg=f)
    np.testing.assert_array_equal(desc, rd)


@pytest.mark.parametrize("total,pageable", [(120000, False), (131072, True)])
def test_outputs_take_the_place_of_inputs(own_ctx, total, pageable):
    """3.84 MB of descriptors in and 0.72 MB of results out: each fits the
    pinned memory, so no copy of pageable memory is made.  4 MiB of
    descriptors leave no room for their offsets."""
    from mcvslam_amd import distinctive_descriptors
    rng = np.random.default_rng(8)
    n = 20000
    ptr = np.concatenate([[0], np.sort(rng.choice(np.arange(1, total), n - 1, replace=False)), [total]])
    desc = rng.integers(0, 256, (total, 32), dtype=np.uint8)
    assert np.diff(ptr).max() <= 256
    got = []
    names = device_events(lambda: got.append(distinctive_descriptors(desc, ptr, ctx=own_ctx)),
                          ["k_copy_parts", "k_distinctive"] + ["Memcpy"] * pageable)
    assert any("k_distinctive" in n for n in names)
    assert any("Memcpy" in n for n in names) == pageable, names
    best, out = got[0]
    want = oracle.distinctive(desc, ptr.astype(np.int32))
    np.testing.assert_array_equal(best, want)
    np.testing.assert_array_equal(out, desc[ptr[:-1] + want])
