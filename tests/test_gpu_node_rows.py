"""The node rows of the FP32 deposit built on the device equal the host builder's, and are built once for a mesh:
clones use them from other streams, before and after the object that built them is gone."""

import numpy as np
import pytest
import torch

import oppx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,order", [(1, "x"), (2, "morton"), (7, "x"), (16, "morton")])
def test_gpu_node_rows_equal_the_host_builder(nx, order):
    m = oppx.box_mesh(nx, nx, nx, order=order)
    pos, vel, p2c = oppx.box_particles(3000, 5, 0.01, m)
    pos, vel, p2c = oppx.sort_particles_by_cell(pos, vel, p2c)
    g = oppx.FempicDevice(m, oppx.box_field_sines(m), pos, vel, p2c)
    dt = 0.2 / nx / 0.01

    def step(d):
        d.step_begin()
        d.pass_fused(1e-3, 1.0, dt)
        d.sort(drop_removed=True)
        return d.deposit_sorted_f32()

    first, other = g.clone(), torch.cuda.Stream()
    with torch.cuda.stream(other):
        want = step(first).cpu().numpy()
    start, ref = oppx.node_cell_csr(dict(n_cells=m["n_cells"], n_nodes=m["n_nodes"], c2n=m["c2n"]))
    assert np.array_equal(first.node_start.cpu().numpy(), start) and np.array_equal(first.node_ref.cpu().numpy(), ref)
    torch.cuda.synchronize()
    rows = first.node_ref.data_ptr()
    del first
    second = g.clone()
    got = step(second).cpu().numpy()
    assert second.node_ref.data_ptr() == rows
    assert np.array_equal(got, want)
