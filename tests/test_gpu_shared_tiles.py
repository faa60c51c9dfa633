"""The projections' shared tiles against fp64 at their edges, through each form of the launch: plain, with the
rotation, and with the rows written into the cache."""
import pytest
import torch

from chunk_attn import capi
import test_gpu_project as project
from test_gpu_project import _close, _draw

pytestmark = pytest.mark.gpu


# shared tiles: 64 x 64, 64 x 128, 128 x 128, 128 x 256 by size, their last rows and columns, one to more stages than
# buffers
@pytest.mark.parametrize("rows,n_out,n_in", [
    (17, 9224, 64), (290, 1024, 64), (512, 2048, 128), (500, 2047, 192), (321, 4096, 256), (700, 4104, 320), (129, 12288, 64),
    (1500, 4096, 448), (2049, 4096, 192), (1023, 8000, 576)])
def test_linear_in_shared_tiles(rows, n_out, n_in):
    g = torch.Generator().manual_seed(rows + n_out)
    x, w = _draw(g, rows, n_in), _draw(g, n_out, n_in, sigma=n_in ** -0.5)
    guard = torch.full((rows * n_out + 64,), 3.0, dtype=torch.float16, device="cuda")
    out = guard[:rows * n_out].view(rows, n_out)
    capi._check(capi.load().ca_linear(x.data_ptr(), w.data_ptr(), out.data_ptr(), rows, n_out, n_in,
                                      torch.cuda.current_stream().cuda_stream))
    _close(out, x.double() @ w.double().t(), n_in)
    assert (guard[rows * n_out:] == 3.0).all()


@pytest.mark.parametrize("n_in", [256, 320, 384])            # one stage less than buffers, as many, one more
def test_linear_in_the_smallest_shared_tiles(n_in):
    test_linear_in_shared_tiles(300, 2050, n_in)


@pytest.mark.parametrize("rows,heads,n_in", [(250, 8, 384), (400, 8, 64), (129, 16, 320), (500, 12, 128), (300, 32, 192), (1030, 31, 256)])
def test_qkv_rotary_in_shared_tiles(rows, heads, n_in):
    project.test_qkv_rotary(rows, heads, n_in)


# tiles of three heads: 128 rows (one to more stages than buffers, last rows, a grid that the XCDs do not divide), 256 rows
# (test_projection_rules holds the rule to these tiles)
@pytest.mark.parametrize("rows,heads,n_in", [(1300, 16, 64), (1409, 16, 128), (1291, 17, 192), (2047, 12, 320),
                                             (1290, 32, 1024), (2000, 31, 1088), (6900, 8, 1024)])
def test_qkv_rotary_in_tiles_of_three_heads(rows, heads, n_in):
    project.test_qkv_rotary(rows, heads, n_in)


def test_decode_of_more_rows_than_a_block():
    project.test_layer_decode_writes_the_pool_as_the_library_path_does(70, 12, 64)


@pytest.mark.parametrize("rows", [20, 70])
def test_linear_beyond_the_reach_of_shared_tiles(rows):
    """2^30 weights and more: 64 x 64 tiles with k split over the waves."""
    n_out, n_in = 16500, 65088
    g = torch.Generator(device="cuda").manual_seed(rows)
    x = torch.randn(rows, n_in, generator=g, device="cuda", dtype=torch.float16)
    w = torch.randn(n_out, n_in, generator=g, device="cuda", dtype=torch.float16).mul_(n_in ** -0.5)
    got = capi.linear(x, w)
    for c in range(0, n_out, 2500):
        _close(got[:, c:c + 2500], x.double() @ w[c:c + 2500].double().t(), n_in)
