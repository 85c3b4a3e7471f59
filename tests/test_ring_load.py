"""What the compiler is told about the direct-to-LDS load in assembly (csrc/ring.h), seen in what it emits around one."""
import importlib
import re
import subprocess

SOURCE = r"""
#include "ring.h"
// The builtin takes its LDS address from m0, too: the same one before and after a load of the ring's.
__global__ void around(const char* a, int bytes, float* out) {
  __shared__ __attribute__((aligned(1024))) char lds[8192];
  const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc((void*)a, 0, bytes, 0x00020000);
  const u32x4 w = {(uint32_t)(uint64_t)a, (uint32_t)((uint64_t)a >> 32), (uint32_t)bytes, 0x00020000u};
  const auto to = (__attribute__((address_space(3))) void*)lds;
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, to, 4, threadIdx.x * 4, 0, 0, 0);
  ring_load(lds_address(lds) + 4096, w, threadIdx.x * 16);
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, to, 4, threadIdx.x * 4, 1024, 256, 0);
  ring_wait<0>();
  out[threadIdx.x] = *(float*)(lds + threadIdx.x * 4);
}
"""


def test_the_compiler_knows_that_a_ring_load_writes_m0(pkg, tmp_path):
    build = importlib.import_module(pkg.__name__ + ".build")
    src, asm = tmp_path / "around.hip", tmp_path / "around.s"
    src.write_text(SOURCE)
    subprocess.run([build.hipcc(), *build.HIPCC_FLAGS, "-I", build.INCLUDE, "-I", build.CSRC, "--cuda-device-only", "-S", str(src),
                    "-o", str(asm)], check=True, capture_output=True)
    seen = [m.group(1) or "m0" for m in re.finditer(r"^\s+(?:s_\w+ m0,.*|(buffer_load_\w+) .*\blds)$", asm.read_text(), re.M)]
    # every load right behind a write of m0
    assert seen == ["m0", "buffer_load_dword", "m0", "buffer_load_dwordx4", "m0", "buffer_load_dword"]
