"""The split-K product of the filter (exh_zgemm_cn_device) over its column
forms: one to eight tiles of eight columns per workgroup and one or two
workgroups across, at the first and last width of each; rows and K that end
inside a tile, a slab and a chunk; C as stored and as its transpose.

Against 64-bit products on the CPU.  Each element is a sum of k products of
standard normals: error <= 8 k eps max|a| max|x|, eps = 2^-53 (four real
products and sums per term, in any order)."""
import pytest


@pytest.mark.gpu
@pytest.mark.parametrize("m", [2, 8, 9, 16, 17, 25, 33, 41, 49, 56, 57, 64, 65, 80, 127, 129])
@pytest.mark.parametrize("nout,k,split", [(67, 203, 1), (130, 61, 0), (16, 9, 4)])
def test_product_widths(m, nout, k, split):
    import torch
    from exciting_amd import lapw
    print(f"[gpu-dense-columns] nout {nout} m {m} k {k} split {split}", flush=True)
    g = torch.Generator().manual_seed(100 * m + k)
    r = lambda *sh: torch.randn(*sh, dtype=torch.complex128, generator=g)
    a, x, y0, z = r(k, nout), r(k, m), r(nout, m), r(nout, m)
    tol = 8 * k * 2.0 ** -53 * a.abs().max().item() * x.abs().max().item() + 1e-15
    got = lapw.zgemm_cn(a.cuda(), x.cuda(), split=split).cpu()
    assert (got - a.conj().t() @ x).abs().max().item() <= tol
    got = lapw.zgemm_cn(a.cuda(), x.cuda(), alpha=0.5, beta=-2.0, y0=y0.cuda(), gamma=3.0,
                        z=z.cuda(), split=split).cpu()
    want = 0.5 * (a.conj().t() @ x) - 2.0 * y0 + 3.0 * z
    assert (got - want).abs().max().item() <= tol + 8 * 2.0 ** -53 * want.abs().max().item()
    if nout == 67:   # conj_a = 0: the row-major transpose of a Hermitian matrix
        c = r(nout, nout)
        c = c + c.conj().t()
        v = r(nout, m)
        got = lapw.zgemm_cn(c.cuda(), v.cuda(), hermitian=True).cpu()
        ct = c.t().contiguous().t().cuda()
        got_t = lapw.zgemm_cn(ct, v.cuda(), hermitian=True).cpu()
        t = 8 * nout * 2.0 ** -53 * c.abs().max().item() * v.abs().max().item()
        assert (got - c @ v).abs().max().item() <= t
        assert (got_t - c @ v).abs().max().item() <= t
