"""BCSC forward scatter over feature widths around its 64-feature steps and
256-feature chunks (a lane holds every 64th feature of a chunk), from
unaligned X and Y too, against the oracle."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("values", [False, True])
@pytest.mark.parametrize("F", [1, 63, 64, 65, 129, 192, 193, 256, 257, 300, 385, 513])
def test_bcsc_scatter_widths(gpu, oracle, F, values):
    _check(oracle, 130, 101, 2500, F, values)


@pytest.mark.parametrize("values", [False, True])
@pytest.mark.parametrize("F", [64, 65, 128, 129, 192, 193, 256, 257, 385])
def test_bcsc_scatter_widths_of_many_waves(gpu, oracle, F, values):
    """Enough blocks for several features a lane."""
    B = _check(oracle, 4000, 2600, 100_000, F, values)
    assert (B.view.num_TCBlocks + 15) // 16 * ((F + 63) // 64) > 4 * 256 or F <= 64


def _check(oracle, nr, nc, nnz, F, values):
    from tcc_amd import swtcf

    rng = np.random.default_rng(F)
    key = np.sort(rng.choice(nr * nc, size=nnz, replace=False))
    dst, src = (key // nc).astype(np.uint32), (key % nc).astype(np.uint32)
    val = rng.standard_normal(nnz).astype(np.float32) if values else None
    X = rng.standard_normal((nc, F)).astype(np.float32)
    Y0 = rng.standard_normal((nr, F)).astype(np.float32)
    B = swtcf.coo_to_bcsc(torch.from_numpy(dst.view(np.int32)).cuda(), torch.from_numpy(src.view(np.int32)).cuda(),
                          None if val is None else torch.from_numpy(val).cuda(), nr, nc)
    rowptr = np.zeros(nr + 1, np.int64)
    np.cumsum(np.bincount(dst, minlength=nr), out=rowptr[1:])
    want = Y0 + oracle.csr_spmm(rowptr, src, val, X, use_tf32=True)
    for shift in (0, 1):  # X and Y aligned to 16 and to 4 bytes, with guard floats around Y
        Xd = torch.empty(nc * F + 1, device="cuda")[shift:shift + nc * F].view(nc, F)
        Xd.copy_(torch.from_numpy(X))
        buf = torch.full((nr * F + 8,), 7.0, device="cuda")
        Yd = buf[shift:shift + nr * F].view(nr, F)
        Yd.copy_(torch.from_numpy(Y0))
        swtcf.bcsc_spmm(B, Xd, Yd)
        # fp32 sums of at most 101 TF32 products a row (4000 rows: 60): well under 101 * 2^-24 of the result
        err = np.linalg.norm(Yd.cpu().numpy() - want) / np.linalg.norm(want)
        assert err <= 6e-6, (F, shift, err)
        assert torch.all(buf[shift + nr * F:] == 7.0)
        assert shift == 0 or buf[0].item() == 7.0
    return B
