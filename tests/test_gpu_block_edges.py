"""The general path's element blocks at the edges of their node loops, against the oracle.

A block's threads load and write its local nodes two at a time; disjoint elements (eight local
nodes each) put a block on either side of one node a thread, two, and of the most it stages.
Tolerances as in test_gpu_operator.py: one apply or diagonal within 1e-12 of the largest entry,
FP32 within 2e-6.
"""
import numpy as np
import pytest

from femorax_amd import core
from oracle import fxo
from tests import meshes

pytestmark = pytest.mark.gpu


def disjoint(count):
    """`count` elements of the distorted box, each with its own eight nodes, the first node fixed."""
    m = meshes.partly_exploded(6, lo=-1.0, hi=2.0)
    keep = np.unique(m["conn"][:count])
    new = np.full(m["nnode"], -1, dtype=m["conn"].dtype)
    new[keep] = np.arange(len(keep))
    m["conn"] = new[m["conn"][:count]]
    m["group"] = m["group"][:count]
    m["xyz"] = m["xyz"][keep]
    m["nnode"] = len(keep)
    m["nelem"] = count
    m["fix"] = np.array([[0, 0], [0, 1], [0, 2]], dtype=m["fix"].dtype)
    return m


@pytest.mark.parametrize("count", [1, 31, 32, 33, 64, 65, 96, 97, 128, 129, 216])
def test_block_node_loops(count):
    model = disjoint(count)
    ctx = core.Context(0)
    pm = core.Mesh(model)
    params = pm.params_for(model)
    batch = core.Batch(ctx, pm, params, fp32=True, general=True)
    om, op = fxo.OracleMesh(model), fxo.elastic_params(params)
    x = meshes.random_vector(pm.neq, 5)
    dx, dy = core.DeviceArray.from_host(ctx, x), core.DeviceArray(ctx, pm.neq)
    kk = (1.0, 40.0, 1.6e3, False)

    def err(got, want):
        return np.max(np.abs(got - want)) / np.max(np.abs(want))

    batch.apply(dx, dy, core.coeffs(*kk))
    assert err(dy.get(), om.apply(op, x, fxo.coeffs(*kk))) <= 1e-12
    batch.diagonal(dy, core.coeffs(*kk))
    assert err(dy.get(), om.diagonal(op, fxo.coeffs(*kk))) <= 1e-12
    x32 = core.DeviceArray.from_host(ctx, x.astype(np.float32), dtype=np.float32)
    y32 = core.DeviceArray(ctx, pm.neq, dtype=np.float32)
    batch.apply_f32(x32, y32)
    assert err(y32.get(), om.apply(op, x.astype(np.float32).astype(np.float64))) <= 2e-6
    ctx.close()
