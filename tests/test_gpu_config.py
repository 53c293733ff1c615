"""The batched kernels' launch configuration: what a fresh context has, and
what a call that leaves the shape alone keeps."""
import pytest

from patchmatch_amd._lib import Context

pytestmark = pytest.mark.gpu


def test_default_shape_is_kept():
    with Context(0) as ctx:
        fresh = ctx.batch_get_config()
        ctx.batch_set_config(use_graph=0)   # a caller who only wants direct launches
        assert ctx.batch_get_config() == dict(fresh, use_graph=0)
        ctx.batch_set_config()
        assert ctx.batch_get_config() == fresh
