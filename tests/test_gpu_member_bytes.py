"""member_bytes, by which the request loop admits members, against what a
resident member holds: its state and diagnostics, the context's scratch
(licom_scratch_bytes) and the context's static 2-D fields (19 FP64 and two
int32 ones)."""
import pytest

import licom_ensemble as le
import licom_tracer as lt

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(96, 64, 30), (128, 96, 55)])
def test_member_bytes_covers_what_a_member_holds(shape, need_gpu):
    c = le.member_case(4100, *shape)
    m = lt.TracerModel(c, precision="mixed")
    held = sum(t.nbytes for d in (m.state, m.diag) for t in d.values()) + m.licomqice.nbytes
    held += m.scratch_bytes() + c.imt * c.jmt * (19 * 8 + 2 * 4)
    m.close()
    said = le.member_bytes(*shape)
    print(f"{shape}: {held} bytes held, {said} estimated", flush=True)
    # the 1-D fields and the SSSNORM partial sums are left out of both sides
    # (tens of kilobytes at most)
    assert held <= said + 32768 and said <= 1.01 * held
