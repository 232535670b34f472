"""backward_fused_kernel's flush in octets: two lanes read a 64-bit LDS cell and clear a half of it each.  Nothing but the order of the two keeps their sums,
so the compiler must be held to it: in the code that it makes of the kernel, a fence stands between the reads and the clears, and a clear is
of a type that may alias the cell's."""
import os
import re
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
SOURCE = """#include "%s"
using namespace dcn;
typedef const Parts<float>::Vec* Ops;
template __global__ void dcn::backward_fused_kernel<3, 4, 4, float>(Params, PlanSet, const unsigned*, const float*, const float*, Ops, const float*, const float*, Ops,
                                                                    const float*, float*, float*, int, unsigned, int, int);
"""


def test_cells_are_read_before_they_are_cleared(tmp_path):
    header = os.path.join(os.path.dirname(HERE), "deform_conv3d_pytorch_op_amd", "csrc", "dcn_backward_fused.h")
    src, out = tmp_path / "flush.hip", tmp_path / "flush.ll"
    src.write_text(SOURCE % header)
    r = subprocess.run([os.environ.get("HIPCC", "/opt/rocm/bin/hipcc"), "--offload-arch=gfx950", "--offload-device-only", "-O1", "-std=c++17", "-munsafe-fp-atomics",
                        "-S", "-emit-llvm", "-w", str(src), "-o", str(out)], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    assert r.returncode == 0, r.stdout
    lines = out.read_text().splitlines()
    tags = dict(re.findall(r"^(!\d+) = !\{(.*)\}$", "\n".join(lines), re.M))
    cells = {m.group(1) for l in lines for m in [re.match(r"\s*(%\d+) = getelementptr .*i64, ptr addrspace\(3\)", l)] if m}
    reads, clears = [], []
    for at, l in enumerate(lines):
        m = re.match(r"\s*%\d+ = load i64, ptr addrspace\(3\) (%\d+),", l)
        if m and m.group(1) in cells:
            reads.append(at)
        m = re.match(r"\s*store i(\d+) 0, ptr addrspace\(3\) (%\d+),.*!tbaa (!\d+)", l)
        if m and m.group(2) in cells and m.group(1) == "32":
            clears.append((at, tags[tags[m.group(3)].split(",")[0]]))
    assert len(clears) == 4                     # channels of a chunk, one voxel of each
    for at, tag in clears:
        assert "omnipotent char" in tag, tag
        last = max(x for x in reads if x < at)
        assert any(re.match(r"\s*fence .*release", l) for l in lines[last:at]) and any(re.match(r"\s*fence .*acquire", l) for l in lines[last:at])
