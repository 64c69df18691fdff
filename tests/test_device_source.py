"""Rules of the device sources that no run shows: the order of LDS accesses
between the lanes of a wavefront."""
import re
from pathlib import Path

CSRC = Path(__file__).resolve().parent.parent / "sphera_amd" / "csrc"


def _code(name):
    return re.sub(r"//[^\n]*", "", (CSRC / name).read_text())


def test_lanes_share_lds_through_fences():
    """wave_barrier() is no memory fence; LDS passes between lanes through
    wave_lds_sync(), which has one on each side."""
    for f in ("sph_kernels.hip", "sph_dbsph.hip"):
        src = _code(f)
        body = re.search(r"void wave_lds_sync\(\) \{(.*?)\n\}", src, re.S)
        if body:
            assert re.fullmatch(r'\s*__builtin_amdgcn_fence\(__ATOMIC_RELEASE, "wavefront"\);'
                                r'\s*__builtin_amdgcn_wave_barrier\(\);'
                                r'\s*__builtin_amdgcn_fence\(__ATOMIC_ACQUIRE, "wavefront"\);\s*', body.group(1))
            src = src.replace(body.group(0), "")
        assert "wave_barrier" not in src, f


def test_list_runs_are_read_as_bytes():
    """The search's list in LDS holds 16- or 32-bit entries and leaves in
    16-byte runs: a run is read as bytes, since a vector type's load may be moved
    before the entries' stores."""
    src = _code("sph_kernels.hip")
    assert not re.search(r"reinterpret_cast<(const )?(uint4|int4)\s*\*>\(list", src)
