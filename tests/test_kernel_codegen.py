"""Code-generation checks of the MFMA GEMM kernels (no GPU needed: hipcc
cross-compiles).  The main-loop MFMAs of the one-wave-per-SIMD kernel are inline
assembly, so the compiler knows neither their latency nor that they are MFMAs;
these tests pin the properties the kernel's correctness argument relies on."""

import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


@pytest.fixture(scope="module")
def gemm_asm(tmp_path_factory):
    if not os.path.exists(HIPCC):
        pytest.skip("hipcc not available")
    out = tmp_path_factory.mktemp("asm") / "gemm_bf16.s"
    src = os.path.join(ROOT, "axonn_amd", "csrc", "gemm_bf16.hip")
    cmd = [HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17", "-Xclang", "-target-feature", "-Xclang",
           "-packed-fp32-ops", "-I" + os.path.join(ROOT, "include"), "-I" + os.path.dirname(src),
           "--cuda-device-only", "-S", src, "-o", str(out)]
    subprocess.run(cmd, check=True, capture_output=True, timeout=900)
    text = out.read_text()
    kernels = {}
    for m in re.finditer(r"^(_ZN3axn\S*gemm_(?:(?:bf16|f16)_(?:solo|rest|swiglu)|backward)_kernel\S*):", text, re.M):
        end = text.index(".end_amdhsa_kernel", m.end())
        kernels[m.group(1)] = text[m.end():end]
    # 7 layout/epilogue/output variants x 3 tile shapes (256 x 256, 128 x 128, 256 x 128) x 2 element
    # types (and the two-term input gradient as an eighth variant), and the gate/up forward of
    # each type
    assert len(kernels) >= 50, sorted(kernels)
    return kernels


def _instructions(body):
    return [ln.split(";")[0].strip() for ln in body.split("\n") if ln.split(";")[0].strip()]


def test_solo_kernels_do_not_spill(gemm_asm):
    for name, body in gemm_asm.items():
        assert re.search(r"\.amdhsa_private_segment_fixed_size 0\b", body), name
        assert "scratch_" not in body, name


def test_accumulators_stay_in_their_registers_until_the_last_mfma_has_retired(gemm_asm):
    """An accumulator copied out of its AGPRs right behind the MFMA that writes it is
    read before the result has left the pipeline.  So: every v_accvgpr_read follows
    the textually preceding MFMA by at least 32 idle cycles (two s_nop 15), and no
    basic block moves AGPRs around (v_accvgpr_mov: the zero-initialisation) behind
    an MFMA of its own."""
    for name, body in gemm_asm.items():
        ins = _instructions(body)
        nops, reads, mfma_in_block = 2, 0, False
        for s in ins:
            if s.startswith(".LBB"):
                mfma_in_block = False
            elif s.startswith("v_mfma"):
                nops, mfma_in_block = 0, True
            elif s == "s_nop 15":
                nops += 1
            elif s.startswith("v_accvgpr_read"):
                assert nops >= 2, (name, s)
                reads += 1
            elif s.startswith("v_accvgpr_mov"):
                assert not mfma_in_block, (name, s)
        assert reads > 0, name


def test_main_loop_mfma_operands_have_fixed_register_classes(gemm_asm):
    """Accumulators in AGPRs, fragments in VGPRs, for every MFMA of every variant."""
    for name, body in gemm_asm.items():
        for s in _instructions(body):
            if s.startswith("v_mfma_f32_16x16x32_"):
                half = "gemm_f16_" in name or "gemm_backward_kernelILb1" in name   # <HALF, ...>
                assert s.split()[0].endswith("_f16" if half else "_bf16"), (name, s)
                ops = [o.strip() for o in s.split(None, 1)[1].split(",")]
                assert ops[0].startswith("a[") and ops[3].startswith("a[") and ops[0] == ops[3], (name, s)
                assert ops[1].startswith("v[") and ops[2].startswith("v["), (name, s)


@pytest.mark.parametrize("source", ["gemm_edge_bf16", "gemm_edge_f16"])
def test_kernels_with_bounds_keep_the_same_properties(tmp_path_factory, source):
    """No spills, and the accumulators' wait behind the last MFMA, also where the stores are
    guarded and the columns behind the last multiple of 8 take another way."""
    kernels = {k: v for k, v in _device_asm(tmp_path_factory, source).items() if "gemm_edge" in k}
    assert len(kernels) >= 29, sorted(kernels)   # 9 layouts and epilogues x 3 tiles, the joint backward x 2
    test_solo_kernels_do_not_spill(kernels)
    test_accumulators_stay_in_their_registers_until_the_last_mfma_has_retired(kernels)
    for body in kernels.values():
        assert "v_mfma_f32_16x16x32_" + source.rsplit("_", 1)[1] in body


_ASM_CACHE = {}


def _device_asm(tmp_path_factory, name):
    if name in _ASM_CACHE:
        return _ASM_CACHE[name]
    if not os.path.exists(HIPCC):
        pytest.skip("hipcc not available")
    out = tmp_path_factory.mktemp("asm") / (name + ".s")
    src = os.path.join(ROOT, "axonn_amd", "csrc", name + ".hip")
    cmd = [HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17", "-Xclang", "-target-feature", "-Xclang",
           "-packed-fp32-ops", "-I" + os.path.join(ROOT, "include"), "-I" + os.path.dirname(src),
           "--cuda-device-only", "-S", src, "-o", str(out)]
    subprocess.run(cmd, check=True, capture_output=True, timeout=900)
    text = out.read_text()
    kernels = {}
    for m in re.finditer(r"^(_ZN\S+):\s", text, re.M):
        end = text.find(".end_amdhsa_kernel", m.end())
        if end > 0 and ".amdhsa_kernel" in text[m.end():end]:
            kernels[m.group(1)] = text[m.end():end]
    _ASM_CACHE[name] = kernels
    return kernels


def _vector_registers(s):
    used = {int(v) for v in re.findall(r"\bv(\d+)\b", s)}
    for a, b in re.findall(r"\bv\[(\d+):(\d+)\]", s):
        used |= set(range(int(a), int(b) + 1))
    return used


def fragments_touched_in_flight(body):
    """(instructions that name a register of an LDS read that may be on its way, number of such reads).  The reads are
    asm statements, and so is the wait for them: nothing tells the compiler that their registers are not written yet.
    Reads stay on their way from one block to the next, so the blocks' ends are followed until nothing is added."""
    blocks, names, in_asm = [[]], {}, False
    for line in body.split("\n"):
        in_asm = (in_asm or "#APP" in line or "#ASMSTART" in line) and "#NO_APP" not in line and "#ASMEND" not in line
        s = line.split(";")[0].strip()
        label = re.fullmatch(r"(\.LBB\w+):", s)
        if label:
            blocks.append([])
            names[label.group(1)] = len(blocks) - 1
        elif s and not s.startswith("."):
            blocks[-1].append((s, in_asm))
            if s.startswith(("s_branch", "s_cbranch", "s_endpgm")):
                blocks.append([])
    found, reads = [], 0
    seen, todo = [None] * len(blocks), [(0, frozenset())]
    while todo:
        at, pending = todo.pop()
        if seen[at] is not None and pending <= seen[at]:
            continue
        seen[at] = pending = pending | (seen[at] or frozenset())
        after = [at + 1]
        for s, asm in blocks[at]:
            assert not s.startswith(("s_setpc", "s_swappc", "s_call")), s
            if s.startswith("s_endpgm"):
                after = []
            elif s.startswith("s_branch"):
                after = [names[s.split()[1]]]
            elif s.startswith("s_cbranch"):
                after = [at + 1, names[s.split()[1]]]
            elif s.startswith("s_waitcnt") and "lgkmcnt(0)" in s:
                pending = frozenset()
            else:
                if _vector_registers(s) & pending:
                    found.append(s)
                if asm and re.match(r"ds_read_b(128|64_tr_b16)\b", s):   # (not the compiler's own reads)
                    reads += 1
                    pending |= _vector_registers(s.split(None, 1)[1].split(",")[0])
        todo += [(b, pending) for b in after if b < len(blocks)]
    return found, reads


def _check_copied_ahead(kernels):
    test_solo_kernels_do_not_spill(kernels)
    test_accumulators_stay_in_their_registers_until_the_last_mfma_has_retired(kernels)
    for name, body in kernels.items():
        found, reads = fragments_touched_in_flight(body)
        assert not found and reads > 0, (name, found[:3])


def test_fragments_in_flight_are_found():
    """What the check below is there for, in a few lines: a register moved in a loop's next turn, or behind a branch."""
    loop = """
.LBB0_1:
  v_mfma_f32_16x16x32_bf16 a[0:3], v[0:3], v[4:7], a[0:3]
  %s
  ;;#ASMSTART
  ds_read_b128 v[0:3], v9
  ;;#ASMEND
  s_cbranch_scc1 .LBB0_1
  s_branch .LBB0_2
.LBB0_2:
  %s
  v_mov_b32_e32 v20, v1
  s_endpgm
"""
    wait = "s_waitcnt lgkmcnt(0)"
    assert fragments_touched_in_flight(loop % (wait, wait))[0] == ["v_mfma_f32_16x16x32_bf16 a[0:3], v[0:3], v[4:7], a[0:3]"]
    loop = loop.replace("  v_mfma", "  s_waitcnt lgkmcnt(0)\n  v_mfma")
    assert fragments_touched_in_flight(loop % ("", wait)) == ([], 2)   # (the loop's block is gone through twice)
    assert fragments_touched_in_flight(loop % ("", "s_waitcnt vmcnt(0)"))[0][0] == "v_mov_b32_e32 v20, v1"


@pytest.mark.parametrize("source,count", [("gemm_fed_rounds", 4), ("gemm_gate_up", 14), ("gemm_fed_nt_bf16", 80),
                                          ("gemm_fed_nt_f16", 80), ("gemm_fed_nn_tn_bf16", 40), ("gemm_fed_nn_tn_f16", 40)])
def test_kernels_with_copying_waves_keep_the_same_properties(tmp_path_factory, source, count):
    """And no instruction touches a fragment before its wait, on any way through the kernel: in gemm_fed_rounds the reads
    of a tile's first fragments are on their way across the end of the loop over the tiles."""
    kernels = {k: v for k, v in _device_asm(tmp_path_factory, source).items() if "gemm_" in k}
    assert len(kernels) == count, sorted(kernels)
    _check_copied_ahead(kernels)


def test_main_loops_touch_no_fragment_before_its_wait(gemm_asm, tmp_path_factory):
    """The same for the kernels of the other two files."""
    for kernels in (gemm_asm, {k: v for k, v in _device_asm(tmp_path_factory, "gemm_edge_bf16").items() if "gemm_edge" in k}):
        for name, body in kernels.items():
            found, reads = fragments_touched_in_flight(body)
            assert not found and reads > 0, (name, found[:3])


def test_stream_kernels_touch_no_fragment_before_its_wait(tmp_path_factory):
    """The forward of a few tokens reads its fragments in asm statements and waits for them in another: until
    then no instruction names their registers."""
    kernels = {k: v for k, v in _device_asm(tmp_path_factory, "gemm_stream").items() if "gemm_stream" in k}
    assert len(kernels) == 108, len(kernels)   # 3 token ranges x 3 heights x 6 epilogues x 2 types
    for name, body in kernels.items():
        assert re.search(r"\.amdhsa_private_segment_fixed_size 0\b", body), name
        pending, reads, in_asm = set(), 0, False
        for line in body.split("\n"):
            in_asm = (in_asm or "#APP" in line or "#ASMSTART" in line) and "#NO_APP" not in line and "#ASMEND" not in line
            s = line.split(";")[0].strip()
            used = {int(v) for v in re.findall(r"\bv(\d+)\b", s)}
            for a, b in re.findall(r"\bv\[(\d+):(\d+)\]", s):
                used |= set(range(int(a), int(b) + 1))
            if in_asm and s.startswith("ds_read_b128"):
                reads += 1
                pending |= set(range(*(int(x) + i for i, x in enumerate(re.search(r"v\[(\d+):(\d+)\]", s).groups()))))
            elif s.startswith("s_waitcnt") and "lgkmcnt(0)" in s:
                pending = set()
            else:
                assert not used & pending, (name, s)
        assert reads > 0, name


def test_gate_up_stream_kernels_touch_no_fragment_before_its_wait(tmp_path_factory):
    """The same for the gate/up forward of a few tokens."""
    kernels = {k: v for k, v in _device_asm(tmp_path_factory, "gemm_stream").items() if "gate_up_stream" in k}
    assert len(kernels) == 16, len(kernels)   # 3 token ranges x 3 heights (up to 16 tokens: 2) x 2 types
    for name, body in kernels.items():
        assert re.search(r"\.amdhsa_private_segment_fixed_size 0\b", body), name
        pending, reads, in_asm = set(), 0, False
        for line in body.split("\n"):
            in_asm = (in_asm or "#APP" in line or "#ASMSTART" in line) and "#NO_APP" not in line and "#ASMEND" not in line
            s = line.split(";")[0].strip()
            used = {int(v) for v in re.findall(r"\bv(\d+)\b", s)}
            for a, b in re.findall(r"\bv\[(\d+):(\d+)\]", s):
                used |= set(range(int(a), int(b) + 1))
            if in_asm and s.startswith("ds_read_b128"):   # (not the compiler's own reads)
                reads += 1
                first, last = map(int, re.search(r"v\[(\d+):(\d+)\]", s).groups())
                pending |= set(range(first, last + 1))
            elif s.startswith("s_waitcnt") and "lgkmcnt(0)" in s:
                pending = set()
            else:
                assert not used & pending, (name, s)
        assert reads > 0, name


@pytest.mark.parametrize("source", ["stream_probe", "embedding"])
def test_hand_written_stores_are_followed_by_their_wait_states(tmp_path_factory, source):
    """A store of more than 8 bytes needs wait states before its data registers are written
    again.  The compiler inserts them for its own stores, not for a store inside an asm
    statement: each of those carries its own s_nop."""
    kernels = _device_asm(tmp_path_factory, source)
    seen = 0
    for name, body in kernels.items():
        ins = _instructions(body)
        for i, s_ in enumerate(ins):
            if s_.startswith("global_store_dwordx4") and "sc1 nt" in s_:
                # (only the asm statements write "sc1 nt"; the compiler prints "nt sc1")
                seen += 1
                assert ins[i + 1].startswith("s_nop"), (name, s_, ins[i + 1])
    assert seen > 0, source


def test_update_kernel_streams_through_buffer_accesses_without_scratch(tmp_path_factory):
    """The optimizer's update kernel: no spills, every streaming access a buffer access with
    its cache policy (loads nt, stores nt sc1), all loads of the vector path ahead of the
    first store."""
    kernels = {k: v for k, v in _device_asm(tmp_path_factory, "optim").items() if "mt_adam_kernel" in k}
    assert len(kernels) == 18, sorted(kernels)   # 3 gradient types x (no copy, bf16, fp16) x with/without scan result
    for name, body in kernels.items():
        assert re.search(r"\.amdhsa_private_segment_fixed_size 0\b", body), name
        ins = _instructions(body)
        loads = [i for i, s_ in enumerate(ins) if s_.startswith("buffer_load_dwordx")]
        stores = [i for i, s_ in enumerate(ins) if s_.startswith("buffer_store_dwordx")]
        assert len(loads) == 4 and len(stores) in (3, 4), (name, len(loads), len(stores))
        assert max(loads) < min(stores), name
        assert all(ins[i].endswith(" nt") for i in loads), name
        assert all(ins[i].endswith(" nt sc1") for i in stores), name


def test_tiles_in_rounds_refuse_columns_that_they_do_not_store(tmp_path):
    """Their epilogue has no LDS for the columns behind the last multiple of 8: the launch refuses such an output, and
    rows that are not 16-byte aligned, whoever calls it."""
    if not os.path.exists(HIPCC):
        pytest.skip("hipcc not available")
    csrc = os.path.join(ROOT, "axonn_amd", "csrc")
    source = tmp_path / "rounds.hip"
    source.write_text("""
        #include <stdio.h>
        #include "gemm_fed_rounds.hip"
        namespace axn {
        void set_error(const char*, ...) {}
        int hip_fail(hipError_t, const char*) { return AXN_EHIP; }
        }
        int main() {
          const int sizes[][2] = {{2060, 2064}, {2056, 2060}, {8, 9}, {7, 8}};
          for (auto& s : sizes) {
            axn::GemmArgs g = {};
            g.M = 8200, g.N = s[0], g.ldc = s[1], g.Kc = 320, g.lda = 8200, g.ldb = 2064;
            printf("%d\\n", axn::launch_gemm_fed_rounds(g, false, axn::FED_128x256, nullptr));
          }
        }""")
    program = tmp_path / "rounds"
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
                    "-I" + os.path.join(ROOT, "include"), "-I" + csrc, str(source), "-o", str(program)],
                   check=True, capture_output=True, timeout=900)
    out = subprocess.run([str(program)], check=True, capture_output=True, text=True, timeout=120).stdout
    assert [int(s) for s in out.split()] == [-3] * 4   # AXN_ESHAPE
