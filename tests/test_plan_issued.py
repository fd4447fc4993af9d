"""What a plan says it issues, without a GPU: the flops of the tiles its launch
runs, which are the trapezoid walk's for either shape and wave tiles for small
products."""
import pytest


def padded(n, m, tm, tn):
    """2 tm tn k over the row tiles, k up to the tile's last row in panels of 16."""
    rows = sum(2.0 * tm * (-(-min(r + tm, n) // 16) * 16) for r in range(0, n, tm))
    return rows * (-(-m // tn) * tn)


@pytest.mark.parametrize("n,m,tm,tn", [
    (257, 257, 16, 16), (1, 1, 16, 16), (1024, 1024, 16, 32), (1600, 1600, 32, 32), (300, 3001, 16, 32),
    (2048, 2048, 64, 64), (4096, 4096, 256, 128), (4099, 2050, 128, 128), (9000, 250, 64, 64),
    (9000, 31, 128, 32), (9000, 16, 16, 16), (28000, 7, 16, 16),
])
def test_issued_flops_are_of_the_launch(uvt, n, m, tm, tn):
    for p, shape in ((1, "trapezoid"), (min(4, n), "boxes")):
        plan = uvt.Plan(n, m, p, "reg", shape)
        assert plan.issued_flops == padded(n, m, tm, tn)
        plan.close()
