"""The inline-assembly steps that broadcast and multiply-add (eight or sixteen
v_fmac with DPP each) write registers while inputs are still to be read: the
compiler must not give an input the register of an in/out operand, which it may
where both hold the same value.  Compiled for gfx950 without a GPU: in the
probes every operand is the same value, and no instruction of a step may read
what an earlier one of the step wrote."""
import re
import subprocess

import pytest

from tmv_amd import build

PROBES = {
    "bcast_fma8": ("tmvx_pivot.h", """
template <typename T, int H> __global__ void probe(T* p)
{
    T r[8];
    const T x = p[threadIdx.x];
    for (int c = 0; c < 8; ++c) r[c] = x;
    bcast_fma8<H, 0>(r, x, x);
    for (int c = 0; c < 8; ++c) p[threadIdx.x + 64 * c] = r[c];
}
template __global__ void probe<double, 0>(double*);
template __global__ void probe<double, 1>(double*);
template __global__ void probe<float, 0>(float*);
template __global__ void probe<float, 1>(float*);
""", 8),
    "zbcast_fma4": ("tmvx_complex_lu.hip", """
template <typename R> __global__ void probe(R* p)
{
    typedef typename CplxT<R>::type Z;
    const R x = p[threadIdx.x];
    Z l[4];
    for (int c = 0; c < 4; ++c) l[c].x = l[c].y = x;
    R xr = x, xi = x;
    zbcast_fma4<0>(xr, xi, x, x, x, l);
    p[threadIdx.x] = xr;
    p[threadIdx.x + 64] = xi;
}
template __global__ void probe<double>(double*);
template __global__ void probe<float>(float*);
""", 16),
}


def registers(op):
    m = re.fullmatch(r"v\[(\d+):(\d+)\]", op)
    if m:
        return set(range(int(m[1]), int(m[2]) + 1))
    return {int(op[1:])}


@pytest.mark.parametrize("name", sorted(PROBES))
def test_inputs_are_not_overwritten(tmp_path, name):
    header, code, count = PROBES[name]
    src, out = tmp_path / "probe.hip", tmp_path / "probe.s"
    src.write_text(f'#include "{header}"\nnamespace tmvx {{{code}}}\n')
    r = subprocess.run([build.HIPCC, *build.FLAGS, "-I", build.CSRC, "--cuda-device-only", "-S",
                        str(src), "-o", str(out)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    steps = 0
    for kernel in re.split(r"^_ZN4tmvx5probe\w*:", out.read_text(), flags=re.M)[1:]:
        ops = re.findall(r"v_fmac_f\d\d_dpp (\S+), (\S+), (\S+) row", kernel.split(".Lfunc_end")[0])
        assert len(ops) == count
        steps += 1
        written = set()
        for dst, a, b in ops:
            assert not (registers(a) | registers(b)) & written, (dst, a, b)
            written |= registers(dst)
    assert steps >= 2
