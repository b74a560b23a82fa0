"""Wait states of the packet gather's compiled code (csrc/kernels/pm_packet.h).

On gfx950 a vector instruction that reads a lane mask (v_cndmask, an add or
subtract with carry-in) must come at least two wait states after the vector
instruction that wrote the mask.  The compiler keeps that distance between its
own instructions and cannot do so across inline assembly.  The test compiles
one instance of the gather to assembly and measures every such pair.
"""
import os
import re
import shutil
import subprocess

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(REPO, "cuda-photon-mapper_amd", "csrc")
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"

SOURCE = """
#include "kernels/pm_packet.h"
namespace pm {
struct Add {
  PowerSum s;
  __device__ void reset() { psum_init(s); }
  __device__ void operator()(V3f pw, V3f, float) { psum_add(s, pw); }
  __device__ Add of_lane(int) const { return *this; }
  __device__ void reduce() { psum_reduce(s); }
  __device__ void take(const Add& o) { s = o.s; }
};
__global__ void __launch_bounds__(64) probe(GatherMap g, const float* q, float* out) {
  __shared__ PacketLds S;
  const int lane = lane_id();
  Add add;
  uint32_t seed = kPkNoSeed, m;
  float r2;
  packet_gather<false>(g, S, lane, true, v3(q[3 * lane], q[3 * lane + 1], q[3 * lane + 2]), seed, add, m, r2);
  out[lane] = (float)add.s.x;
}
}  // namespace pm
"""

MASK = r"(s\[\d+:\d+\]|vcc)"
# a vector instruction's written mask, and the mask it reads
WRITES = [re.compile(r"v_cmp\w+ " + MASK + ","), re.compile(r"v_(?:add|sub|subrev|addc|subb|subbrev)_co_u32\w* v\d+, " + MASK + ",")]
READS = re.compile(r"v_(?:cndmask_b32|addc_co_u32|subb_co_u32|subbrev_co_u32)\w* .*, " + MASK + "$")


def mask_distances(asm):
    """Wait states between the write of a mask and its next read, within straight-line code."""
    out, written, at = [], {}, 0
    for line in asm.splitlines():
        s = line.split(";")[0].strip()
        if not s or s.startswith((".", "//")) or s.endswith(":"):
            if s.endswith(":"):
                written = {}
            continue
        m = READS.match(s)
        if m and m.group(1) in written:
            out.append((at - written[m.group(1)] - 1, s))
        for w in WRITES:
            m = w.match(s)
            if m:
                written[m.group(1)] = at
        if s.startswith("s_"):  # a scalar instruction's own write is another kind of mask
            for m in re.findall(MASK, s.split(",")[0]):
                written.pop(m, None)
        at += 1 + (int(s.split()[1]) if s.startswith("s_nop") else 0)
    return out


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="needs hipcc")
def test_masks_are_read_two_wait_states_after_they_are_written(tmp_path):
    src, asm = tmp_path / "probe.hip", tmp_path / "probe.s"
    src.write_text(SOURCE)
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17", "-ffp-contract=off", "-fno-fast-math",
                    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-w", "--cuda-device-only", "-S",
                    "-I", CSRC, "-o", str(asm), str(src)], check=True)
    d = mask_distances(asm.read_text())
    assert len(d) > 50  # the kernel was found, and its masks
    short = [x for x in d if x[0] < 2]
    assert not short, "%d of %d masks are read too early, such as %s" % (len(short), len(d), short[0])
