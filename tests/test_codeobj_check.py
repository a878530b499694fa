"""Build-time guard for the untracked LDS DMA of the packed-weight MoE kernels.

The pipelines in csrc/w4pk.h issue ``buffer_load ... lds`` as inline assembly
that the compiler's wait pass does not see, which is only correct while those
kernels use no scratch (a spill reload's wait would reorder the DMA) and while
the assembly keeps its hazard padding. These CPU tests compile small kernels
with hipcc (no GPU) and check that ``intent_amd.build.build`` rejects the bad
ones and passes the library's own objects.
"""
import shutil
from pathlib import Path

import pytest

from intent_amd import build as B
from intent_amd import codeobj_check as C

pytestmark = pytest.mark.skipif(shutil.which(B.hipcc()) is None and not Path(B.hipcc()).exists(),
                                reason="hipcc not available")

_CSRC = str(B.CSRC)

# A kernel named like a registered untracked-DMA kernel, using the library's
# own assembly DMA, with a VGPR budget small enough to force spills.
_SPILLING = r'''
#include "mfma_pipe.h"
extern "C" __global__ __attribute__((amdgpu_num_vgpr(24))) __launch_bounds__(256)
void moe_gate_up_pk_kernel_spill_case(const float* __restrict__ p, int n, float* __restrict__ out) {
  __shared__ float buf[4096];
  mp::Rsrc rs = make_rsrc(p);
  float acc[48];
#pragma unroll
  for (int i = 0; i < 48; ++i) acc[i] = p[threadIdx.x + 256 * i];
  for (int it = 0; it < n; ++it) {
    mp::lds_dma<16, true>(rs, (mp::lds_t*)(buf + 256 * (it & 3)), threadIdx.x * 16, it * 4096);
#pragma unroll
    for (int i = 0; i < 48; ++i) acc[i] = acc[i] * acc[(i + 7) % 48] + buf[(threadIdx.x + i) & 4095];
    __syncthreads();
  }
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < 48; ++i) s += acc[i];
  out[threadIdx.x] = s;
}
'''

# The same DMA with no register pressure: accepted.
_CLEAN = r'''
#include "mfma_pipe.h"
extern "C" __global__ __launch_bounds__(256)
void moe_gate_up_pk_kernel_clean_case(const float* __restrict__ p, int n, float* __restrict__ out) {
  __shared__ float buf[4096];
  mp::Rsrc rs = make_rsrc(p);
  for (int it = 0; it < n; ++it) {
    mp::lds_dma<16, true>(rs, (mp::lds_t*)(buf + 1024 * (it & 3)), threadIdx.x * 16, it * 4096);
    mp::wait_vm<0>();
    __syncthreads();
  }
  out[threadIdx.x] = buf[threadIdx.x];
}
'''

# Assembly DMA written without the M0 wait state: rejected.
_NO_NOP = r'''
#include "mfma_pipe.h"
extern "C" __global__ __launch_bounds__(256)
void m0_hazard_case(const float* __restrict__ p, int n, float* __restrict__ out) {
  __shared__ float buf[1024];
  mp::Rsrc rs = make_rsrc(p);
  for (int it = 0; it < n; ++it) {
    const uint32_t m = (uint32_t)(uintptr_t)(mp::lds_t*)(buf + 64 * (it & 3));
    asm volatile("s_mov_b32 m0, %0\n\tbuffer_load_dword %1, %2, %3 offen lds"
                 : : "s"(m), "v"(threadIdx.x * 4), "s"(rs), "s"(it * 256) : "memory");
  }
  mp::wait_vm<0>();
  __syncthreads();
  out[threadIdx.x] = buf[threadIdx.x];
}
'''


def _build(tmp_path, name, text):
    src = tmp_path / f"{name}.hip"
    src.write_text(text)
    return B.build(sources=[src], extra_flags=[f"-I{_CSRC}"], library=tmp_path / f"lib{name}.so",
                   objdir=tmp_path / name)


def test_spilling_untracked_dma_kernel_is_rejected(tmp_path):
    with pytest.raises(C.CodeObjectError, match="spill|scratch|private segment"):
        _build(tmp_path, "spill", _SPILLING)


def test_clean_untracked_dma_kernel_builds(tmp_path):
    lib = _build(tmp_path, "clean", _CLEAN)
    assert lib.exists()


def test_missing_m0_wait_state_is_rejected(tmp_path):
    with pytest.raises(C.CodeObjectError, match="M0"):
        _build(tmp_path, "nonop", _NO_NOP)


def test_library_packed_moe_kernels_pass_the_check(tmp_path):
    """The library's own moe.hip: its packed-weight kernels are found, carry
    LDS DMA and pass (no scratch, padded hazards)."""
    obj = B._compile(B.CSRC / "moe.hip", tmp_path)
    reports = C.check_binary(obj, tmp_path / "co")
    for k in C.UNTRACKED_DMA_KERNELS:
        found = [r for r in reports if k in r.name]
        assert found, k
        assert all(r.dma > 0 and r.spills == 0 and r.private_segment == 0 and r.scratch_ops == 0 for r in found)


def test_valu_sgpr_write_parser():
    assert C._valu_sgpr_writes("v_readfirstlane_b32 s7, v3") == {"s7"}
    assert C._valu_sgpr_writes("v_cmp_gt_i32_e32 vcc, s6, v11") == {"vcc"}
    assert C._valu_sgpr_writes("v_mad_u64_u32 v[20:21], s[2:3], v11, s10, v[20:21]") == {"s2", "s3"}
    assert C._valu_sgpr_writes("v_or_b32_e32 v11, s7, v9") == set()
    assert C._dma_sgpr_reads("buffer_load_dwordx4 v8, s[24:27], s2 offen lds") == {"s24", "s25", "s26", "s27", "s2"}


# An MFMA whose fragment is read from LDS in only the lanes of rows below M: the shape a compiler that moves the
# last fragment read into an epilogue's branch would leave. MFMAs ignore EXEC, the read does not.
_MASKED_OPERAND = r'''
#include "mfma_pipe.h"
extern "C" __global__ __launch_bounds__(64)
void masked_operand_case(const f16* __restrict__ p, int M, float* __restrict__ out) {
  __shared__ __attribute__((aligned(16))) f16 buf[64 * 16];
  const int lane = threadIdx.x;
  for (int i = 0; i < 16; ++i) buf[lane * 16 + i] = p[lane * 16 + i];
  __syncthreads();
  f16x8 a = *reinterpret_cast<const f16x8*>(buf + lane * 16), b = *reinterpret_cast<const f16x8*>(buf + lane * 16 + 8);
  f32x16 acc{};
  SETTLED
  if (lane < M) {
    FRAGMENT
    acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, acc, 0, 0, 0);
    for (int i = 0; i < 16; ++i) out[lane * 16 + i] = acc[i];
  }
}
'''


def test_fragment_read_under_a_mask_is_rejected(tmp_path):
    text = _MASKED_OPERAND.replace("SETTLED", "").replace(
        "FRAGMENT", "a = *reinterpret_cast<const f16x8*>(buf + ((lane * 16 + M * 8) & 1023)); asm volatile(\"\" : \"+v\"(a));")
    with pytest.raises(C.CodeObjectError, match="lanes masked off"):
        _build(tmp_path, "masked", text)


def test_fragments_read_by_the_whole_wave_build(tmp_path):
    text = _MASKED_OPERAND.replace("SETTLED", "asm volatile(\"\" : \"+v\"(a), \"+v\"(b));").replace("FRAGMENT", "")
    assert _build(tmp_path, "whole", text).exists()


def _listing(text):
    """(address, text, branch target) of a listing with one instruction per line; 'label:' names the next one."""
    lines, labels = [], {}
    for line in (x.strip() for x in text.strip().splitlines()):
        if line.endswith(":"):
            labels[line[:-1]] = len(lines) * 4
        else:
            lines.append(line)
    return [(i * 4, s, labels.get(s.split()[-1]) if s.startswith(("s_branch", "s_cbranch")) else None)
            for i, s in enumerate(lines)]


_MFMA = "v_mfma_f32_32x32x16_f16 a[0:15], v[10:13], v[14:17], a[0:15]"
_PIECES = {"read": "ds_read_b128 v[10:13], v0", "shift": "v_bfe_u32 v16, v2, v4, 8", "mfma": _MFMA,
           "mask": "s_and_saveexec_b64 s[2:3], vcc\ns_cbranch_execz end", "end": "end:\ns_or_b64 exec, exec, s[2:3]"}


@pytest.mark.parametrize("order,bad", [
    ("read shift mfma mask end", 0), ("read shift mask mfma end", 0), ("mask read mfma end", 1),
    ("read mask shift mfma end", 1), ("mask read end read mfma", 0), ("read mask mfma shift mfma end", 1)])
def test_masked_operands_of_a_branch(order, bad):
    text = "\n".join(_PIECES[p] for p in order.split())
    found = C.masked_mfma_operands(_listing(text + "\ns_endpgm"))
    assert len(found) == bad, found


def test_masked_operands_of_nested_branches_and_loops():
    # an inner mask restored by the outer one, the other side of a branch, and lanes leaving a loop
    nested = """
      s_and_saveexec_b64 s[2:3], vcc
      s_cbranch_execz out
      s_and_saveexec_b64 s[4:5], s[6:7]
      s_xor_b64 s[4:5], exec, s[4:5]
      s_cbranch_execz other
      ds_read_b128 v[10:13], v0
    other:
      s_andn2_saveexec_b64 s[4:5], s[4:5]
      s_cbranch_execz out
      %s
    out:
      s_or_b64 exec, exec, s[2:3]
      %s
      s_endpgm
    """
    assert C.masked_mfma_operands(_listing(nested % ("v_nop", _MFMA))) == []
    assert len(C.masked_mfma_operands(_listing(nested % (_MFMA, "v_nop")))) == 1
    loop = """
    top:
      ds_read_b128 v[10:13], v0
      %s
      v_cmp_lt_i32_e32 vcc, v1, v2
      s_or_b64 s[2:3], vcc, s[2:3]
      s_andn2_b64 exec, exec, s[2:3]
      s_cbranch_execnz top
      s_or_b64 exec, exec, s[2:3]
      %s
      s_endpgm
    """
    assert len(C.masked_mfma_operands(_listing(loop % (_MFMA, "v_nop")))) == 1  # from its second pass on
    assert C.masked_mfma_operands(_listing(loop % ("v_nop", _MFMA))) == []
