"""The solve's statistics on both sides of the line between one workgroup a channel
and the general kernels (64 tiles): the same bits alone and beside a large channel."""
import pytest

from tests.test_gpu_stats import test_statistics_do_not_depend_on_the_path as check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("solver", ["rb", "lex"])
@pytest.mark.parametrize("nx,ny", [(252, 64), (253, 64), (256, 64), (257, 64), (128, 65), (129, 65),
                                   (13, 1000), (21, 670), (64, 256), (64, 257)])
def test_statistics_around_the_line(nx, ny, solver):
    check(nx, ny, solver)
