"""Rules by size, on the CPU. The forward projection's kernel: the line sweep walks lines of both directions, so narrow
images, whose longer side costs the walk and whose few pixels cost the table little, keep the table. The block products'
split: launches of few waves are split finer, for the walk is all there is."""
import pytest

from diffractom_amd.operator import SinglePhaseForwardOperator

LINES = [(99, 99, 18, 64), (128, 128, 18, 64), (256, 256, 6, 3008), (100, 50, 18, 2048), (200, 64, 18, 9920),
         (84, 42, 90, 9920), (64, 64, 60, 2048), (64, 32, 90, 9920), (256, 102, 18, 64), (81, 60, 1, 64)]
TABLE = [(256, 8, 18, 2048), (256, 8, 180, 9920), (128, 16, 18, 576), (16, 128, 18, 576), (99, 24, 18, 9920),
         (256, 32, 90, 576), (128, 51, 18, 2048), (64, 32, 18, 9920), (72, 36, 18, 9920), (32, 32, 18, 512),
         (72, 72, 18, 512), (1, 1, 1, 64), (257, 8, 18, 2048)]


@pytest.mark.parametrize("nx,ny,n_angles,kn,kernel", [(*c, "lines") for c in LINES] + [(*c, "table") for c in TABLE])
def test_kernel_by_size(nx, ny, n_angles, kn, kernel):
    op = object.__new__(SinglePhaseForwardOperator)
    op.Nx, op.Ny, op.radon_bands = nx, ny, 1
    assert op._fwd_kernel({"pairs_ok": True}, n_angles, kn) == kernel
    assert op._fwd_kernel({"pairs_ok": False}, n_angles, kn) == "table"
    assert op._fwd_kernel(None, n_angles, kn) == "table"


@pytest.mark.parametrize("my,n_ang,n_jb,n_kb,ks", [
    (32, 3, 4, 17, 8), (103, 1, 12, 17, 8), (103, 10, 4, 17, 8), (32, 18, 4, 10, 5), (103, 10, 29, 7, 1), (103, 1, 4, 7, 1),
    (103, 18, 29, 17, 1), (103, 18, 29, 47, 3), (103, 18, 29, 94, 7), (103, 18, 29, 929, 16), (131, 9, 29, 17, 1),
    (131, 9, 8, 17, 7), (17, 1, 1, 1, 1), (17, 1, 1, 3, 1), (17, 1, 1, 7, 1), (17, 1, 1, 8, 4), (17, 1, 1, 5000, 64)])
def test_block_product_split(my, n_ang, n_jb, n_kb, ks):
    op = object.__new__(SinglePhaseForwardOperator)
    op.My, op.blk_variant = my, {}
    assert op._blk_split(n_ang, {"n_jb": n_jb, "n_kb": n_kb}) == ks
