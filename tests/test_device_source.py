"""Rules of the device sources that no run shows: the order of LDS accesses
between the lanes of a wavefront, integer positions across their wrap."""
import re
import subprocess
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


WRAP = r"""
#define __host__
#define __device__
#include "sph_device.h"
#include <cstdio>
static int at(long long u) { return (int)(uint32_t)((unsigned long long)u & 0xFFFFFFFFull); }
int main() {
    const long long cell = 1ll << 28;
    long long n = 0;
    // particles of a grid of 64 cells, two cells apart at most, on both sides of every wrap
    for (long long c = 0; c < 64; ++c)
        for (long long o = -3; o <= 3; ++o)
            for (long long d = -2 * cell - 5; d <= 2 * cell + 5; d += cell / 3 + 1) {
                const long long a = c * cell + o, b = a + d;
                if (b < 0) continue;
                if (sph::lsb_diff(at(a), at(b)) != a - b || sph::lsb_diff(at(b), at(a)) != b - a) return 1;
                ++n;
            }
    std::printf("%lld pairs\n", n);
    return n > 1000 ? 0 : 2;
}
"""


def test_integer_positions_wrap_without_overflow(tmp_path):
    """Separations across a wrap of the integer positions, under the
    undefined-behaviour sanitizer on the CPU; the kernels form every
    separation with that one function."""
    src = tmp_path / "wrap.cpp"
    src.write_text(WRAP)
    exe = tmp_path / "wrap"
    subprocess.run(["g++", "-std=c++17", "-O1", "-w", "-fsanitize=undefined", "-fno-sanitize-recover=all",
                    "-I", str(CSRC), str(src), "-o", str(exe)], check=True)
    subprocess.run([str(exe)], check=True)
    code = _code("sph_kernels.hip")
    assert len(re.findall(r"\(float\)lsb_diff\(", code)) >= 12
    # no signed difference of positions turned into a float
    assert not re.findall(r"\(float\)\(\w+\.[xyz] - (?:\w+\.[xyz]\b|__float_as_int)", code)


WALKS = r"""
#define __host__
#define __device__
#include "sph_device.h"
int main() {
    // the FP32 walk of a gathering particle i reads the groups 0 and 1 of its list,
    // whatever its length, before it looks at the length
    for (int mj = 1; mj <= 100; ++mj)
        for (size_t N = 1; N <= 300; N += 23)
            for (size_t i = 0; i < N; ++i)
                for (size_t m = 0; m < 2; ++m)
                    if ((m * N + i + 1) * sph::NB_G > N * (size_t)sph::nb_stride(mj)) return 1;
    for (int mj = 1; mj <= 1000; ++mj)
        if (sph::nb_stride(mj) < mj || sph::nb_stride(mj) % sph::NB_G) return 2;
    return 0;
}
"""


def test_first_groups_of_a_list_are_in_range(tmp_path):
    (tmp_path / "walks.cpp").write_text(WALKS)
    exe = tmp_path / "walks"
    subprocess.run(["g++", "-std=c++17", f"-I{CSRC}", str(tmp_path / "walks.cpp"), "-o", str(exe)], check=True)
    assert subprocess.run([str(exe)]).returncode == 0
