"""A persistent work queue that runs dry while its workgroup 0 still offers forks."""
import ctypes

import pytest
from test_gpu_kernel_merge import Chunks, km, reduce_buffers  # noqa: F401

from gpu_workgroup_managment_amd import _lib as L
from gpu_workgroup_managment_amd import scheduler as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tasks", [0, 1, 3])
def test_work_queue_ends_without_tasks(rt, km, dev, tasks):  # noqa: F811
    """Members that find the queue empty return and are free again while others
    work on: no fork may take them for workgroups above the persistent range."""
    length, d_buf, d_res, d_calls = reduce_buffers(dev)
    c = Chunks(dev, rounds=16)
    args = L.Args([ctypes.c_int32(length), d_buf.ptr, d_res.ptr, d_calls.ptr] + c.args())
    with S.Mega(rt, np_kind=S.NP_REDUCE_MIN) as m:
        p = m.launch_custom(km.km_mega_chunks(), args, wg_size=256, num_wgs=16)
        m.send_persistent_custom(p)
        for k in range(tasks):
            if m.persistent_running():
                m.send_task_custom(1 + k)
        m.wait_persistent(20)
        m.quit()
    c.check()
    c.free()
    for d in (d_buf, d_res, d_calls):
        d.free()
