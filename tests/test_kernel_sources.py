"""Rules of the kernel sources that no run can show."""
import re
from pathlib import Path

CSRC = Path(__file__).resolve().parent.parent / "openaerolab_alpha_01_amd" / "csrc"


def test_lds_exchange_within_a_wave_is_fenced():
    """Lanes of a wave that read each other's LDS words do so behind wave_sync(): a scheduling barrier between a
    release and an acquire fence.  A bare barrier orders no memory access."""
    sources = {p.name: p.read_text() for p in sorted(CSRC.glob("*.h")) + sorted(CSRC.glob("*.hip"))}
    body = re.search(r"void wave_sync\(\) \{(.*?)\n\}", sources["oal_device.h"], re.S)
    assert body, "wave_sync() is gone"
    order = [body.group(1).find(s) for s in ("__ATOMIC_RELEASE", "amdgcn_wave_barrier", "__ATOMIC_ACQUIRE")]
    assert -1 not in order and order == sorted(order), order
    for name, text in sources.items():
        rest = text.replace(body.group(0), "") if name == "oal_device.h" else text
        assert "amdgcn_wave_barrier" not in rest, name
