"""CPU-only checks of the host side: the library loads and exports every symbol
the C header declares, the prepacked cache follows the reference's known
answers, the ruy:: headers accept the reference's own example programs, and
the Python mirror has the reference's defaults. No device computation here."""
import ctypes as C
import os
import re
import shutil
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "ruy_amd", "c_api.h")
LIB = os.path.join(ROOT, "ruy_amd", "libruy_amd.so")
REFERENCE = "/root/reference"


def declared_symbols():
    text = open(HEADER).read()
    return sorted(set(re.findall(r"RUYAMD_API\s+[^;(]*?\b(ruyamd_\w+)\s*\(", text)))


def test_library_exports_every_declared_symbol():
    assert os.path.exists(LIB), "build the library first: python -m ruy_amd.build"
    lib = C.CDLL(LIB)
    names = declared_symbols()
    assert len(names) >= 25
    for name in names:
        assert hasattr(lib, name), "libruy_amd.so lacks %s" % name
    lib.ruyamd_version.restype = C.c_char_p
    assert b"gfx950" in lib.ruyamd_version()


def test_python_binding_covers_the_header():
    from ruy_amd import _capi
    assert sorted(_capi.PROTOTYPES) == declared_symbols()


def test_struct_layouts_match_the_header():
    """ctypes mirrors vs the C compiler's view of ruyamd_mat / ruyamd_mul_params."""
    from ruy_amd import _structs as S
    src = r'''
#include <stdio.h>
#include <stddef.h>
#include "ruy_amd/c_api.h"
int main(void) {
  printf("%zu %zu %zu %zu %zu %zu %zu %zu\n", sizeof(ruyamd_mat), offsetof(ruyamd_mat, rows),
         offsetof(ruyamd_mat, zero_point), offsetof(ruyamd_mat, order), offsetof(ruyamd_mat, cache_policy),
         sizeof(ruyamd_mul_params), offsetof(ruyamd_mul_params, clamp_min),
         offsetof(ruyamd_mul_params, accum_dtype));
  return 0;
}'''
    work = os.path.join(ROOT, "tests", "cpp", "_layout_probe")
    with open(work + ".c", "w") as f:
        f.write(src)
    try:
        subprocess.check_call(["gcc", "-I" + os.path.join(ROOT, "include"), work + ".c", "-o", work])
        got = [int(x) for x in subprocess.check_output([work]).split()]
    finally:
        for ext in ("", ".c"):
            if os.path.exists(work + ext):
                os.remove(work + ext)
    want = [C.sizeof(S.Mat), S.Mat.rows.offset, S.Mat.zero_point.offset, S.Mat.order.offset,
            S.Mat.cache_policy.offset, C.sizeof(S.MulParamsStruct),
            S.MulParamsStruct.clamp_min.offset, S.MulParamsStruct.accum_dtype.offset]
    assert got == want


def test_prepacked_cache_known_answers():
    """ruy/prepacked_cache_test.cc:54-227 restated over the host-side cache class."""
    exe = os.path.join(ROOT, "tests", "cpp", "prepacked_cache_test")
    subprocess.check_call(["g++", "-std=c++17", "-I" + os.path.join(ROOT, "ruy_amd", "csrc"),
                           exe + ".cc", os.path.join(ROOT, "ruy_amd", "csrc", "prepacked_cache.cc"),
                           "-o", exe])
    out = subprocess.check_output([exe]).decode()
    assert "all passed" in out


def test_host_launch_arithmetic():
    """Grid shapes stay inside HIP's limits and still cover every element."""
    exe = os.path.join(ROOT, "tests", "cpp", "host_logic_test")
    subprocess.check_call(["g++", "-std=c++17", "-pthread", "-I" + os.path.join(ROOT, "ruy_amd", "csrc"),
                           exe + ".cc", "-o", exe])
    out = subprocess.check_output([exe]).decode()
    assert "all passed" in out


def test_ring_schedule_of_the_largest_tile_model():
    """The positions of the matrix instructions, fragment reads, loads and
    barriers of the 256x256 int8 tile's ring step (kernels/paired_schedule.h,
    which the kernel is generated from), run through a host model of registers,
    LDS and barriers; the model must also refuse a list of altered schedules."""
    exe = os.path.join(ROOT, "tests", "cpp", "paired_schedule_test")
    subprocess.check_call(["g++", "-std=c++17", "-I" + os.path.join(ROOT, "ruy_amd", "csrc"),
                           exe + ".cc", "-o", exe])
    out = subprocess.check_output([exe]).decode()
    assert "all passed" in out
    assert out.count("altered (") >= 12


def kernel_assembly(tmp_path, source):
    """The instructions of the first kernel of a source file whose name holds a text."""
    from ruy_amd import build
    asm = str(tmp_path / "kernels.s")
    subprocess.check_call([build.HIPCC] + build.COMMON + build.DEVICE + [
        "--offload-device-only", "-S", os.path.join(build.CSRC, "kernels", source), "-o", asm])
    lines = [l.split(";")[0].strip() for l in open(asm)]

    def body(name):
        start = next(i for i, l in enumerate(lines) if name in l and l.endswith(":"))
        return lines[start:next(i for i in range(start, len(lines)) if lines[i].startswith(".Lfunc_end"))]
    return body


def test_a_lane_of_a_row_pack_has_four_loads_in_flight(tmp_path):
    """Rows of 16 and of 64 lanes: none of a lane's four loads is awaited before
    the last of them is issued."""
    body = kernel_assembly(tmp_path, "pack.hip")
    for kernel in ("PackKernelILi1ELi0E", "PackKernelILi2ELi0E"):
        steps = "".join("L" if l.startswith("global_load_dwordx4") else
                        "w" if l.startswith("s_waitcnt") and "vmcnt" in l else "" for l in body(kernel))
        assert "LLLL" in steps and steps.count("L") == 4, (kernel, steps)


def test_loads_of_the_small_tiles_claim_no_alignment_they_lack(tmp_path):
    """Rows at multiples of 4 bytes whose length is none, and counts that are none:
    the 16 bytes that end with them start anywhere, and the type of such a load has
    to say so. (fp32 lies at multiples of 4 bytes throughout.) It is one load all
    the same."""
    from ruy_amd import build
    source = tmp_path / "fetch.hip"
    source.write_text("""
#include "kernels/mfma_gemm.h"
#include "kernels/small_gemm.h"
namespace ruyamd {
namespace small_gemm {
template <int kSource, int kElement>
__global__ void Fetch(const char* data, int pitch, int count, int bytes, int step, v4i* out) {
  using S = Side<32, 64, kSource, kElement>;
  S side;
  side.Start(data, pitch, count, 0, bytes, 0, threadIdx.x);
  typename S::Held held = {};
  side.Load(step, held);
  for (int u = 0; u < S::kUnits; ++u)
    for (int j = 0; j < S::kLoads; ++j) out[(u * S::kLoads + j) * 64 + threadIdx.x] = held.x[u][j];
}
""" + "".join("template __global__ void Fetch<%d, %d>(const char*, int, int, int, int, v4i*);\n" % (form, element)
              for form in (0, 2) for element in (1, 2, 4)) + "}\n}\n")
    flags = [build.HIPCC] + build.COMMON + build.DEVICE + ["--offload-device-only", "-S", str(source), "-o"]
    subprocess.check_call(flags + [str(tmp_path / "fetch.ll"), "-emit-llvm"])
    claims, name = {}, None
    for line in open(tmp_path / "fetch.ll"):
        if line.startswith("define "):
            name = re.search(r"FetchILi(\d)ELi(\d)E", line).groups()
        if re.search(r" = load <4 x i32>, ptr addrspace\(1\)", line):
            claims.setdefault(name, set()).add(int(re.search(r"align (\d+)", line).group(1)))
    assert claims == {(source, element): {4 if element == "4" else 1} for source in "02" for element in "124"}, claims
    subprocess.check_call(flags + [str(tmp_path / "fetch.s")])
    loads = [line.split()[0] for line in open(tmp_path / "fetch.s") if line.strip().startswith(("global_load", "flat_load"))]
    assert loads and set(loads) == {"global_load_dwordx4"}, loads


def test_every_wave_of_a_download_awaits_its_stores(tmp_path):
    """The word that tells the host a workgroup's part of a download is there is
    stored by one wave (kernels/host_copy.hip). A workgroup barrier by itself
    waits for no store on this target, so each wave has to write back and await
    its own in front of it: looked up in the assembly, between the last store of
    the copy and the barrier."""
    body = kernel_assembly(tmp_path, "host_copy.hip")("DownloadKernel")
    barrier = body.index("s_barrier")
    last_store = max(i for i, l in enumerate(body[:barrier]) if l.startswith("global_store_dwordx4"))
    between = body[last_store + 1:barrier]
    write_back = [i for i, l in enumerate(between) if re.match(r"buffer_wbl2\s+sc0 sc1", l)]
    awaited = [i for i, l in enumerate(between) if l.startswith("s_waitcnt") and "vmcnt(0)" in l]
    assert write_back and awaited and awaited[-1] > write_back[-1], between
    # ... and every wave gets there: the copy's own bounds tests have ended.
    assert any(l.startswith("s_or_b64 exec, exec") for l in between[:write_back[-1]]), between
    flag = [i for i, l in enumerate(body) if re.match(r"global_store_dword\s", l)]
    assert len(flag) == 1 and flag[0] > barrier, flag


def test_no_load_is_on_its_way_to_lds_when_partial_sums_are_put_there(tmp_path):
    """The 64x64 tile of fp32 gives every wave a ring of its own, whose memory the
    waves' partial sums go to behind a workgroup barrier. The barrier does not wait for
    loads that write to LDS, and on bf16 parts the last trip of the loop asks for a step
    past the end (zeros): followed along the branches of the assembly, no path from
    such a load to a barrier is without a wait for all of them."""
    body = kernel_assembly(tmp_path, "gemm_f32.hip")("F32TraitsELi1ELi1ELi128ELi4ELb0ELb0ELb1E")
    labels = {l[:-1]: i for i, l in enumerate(body) if l.endswith(":")}
    loads = [i for i, l in enumerate(body) if l.startswith("buffer_load_dwordx4") and l.endswith(" lds")]
    assert loads and any(l.startswith("v_mfma_f32_32x32x16_bf16") for l in body) and "s_barrier" in body
    on_their_way, seen = [i + 1 for i in loads], set()
    while on_their_way:
        i = on_their_way.pop()
        if i in seen or i >= len(body):
            continue
        seen.add(i)
        l = body[i]
        assert l != "s_barrier", body[max(0, i - 12):i + 1]
        if l.startswith("s_endpgm") or l.startswith("s_waitcnt") and "vmcnt(0)" in l:
            continue
        branch = re.match(r"s_c?branch\w*\s+(\S+)", l)
        if branch:
            on_their_way.append(labels[branch.group(1)])
        if not l.startswith("s_branch"):
            on_their_way.append(i + 1)


def test_matrix_instructions_written_as_text_keep_their_distances(tmp_path):
    """v_mfma_f32_32x32x16_bf16 and v_mfma_i32_16x16x64_i8 stand in the larger kernels as
    assembler text, which the compiler keeps no distances to: two wait states behind a
    vector instruction that writes one of its operands, and 12 or 8 (eight and four
    passes) in front of anything but a matrix instruction that touches its result. The
    compiler is free to copy or clear an accumulator anywhere, so both are looked for
    along the branches of these kernels as they were built."""
    from ruy_amd import build
    objdump = os.path.join(os.path.dirname(os.path.dirname(build.HIPCC)), "llvm", "bin", "llvm-objdump")
    shutil.copy(LIB, tmp_path / "library.so")
    subprocess.check_call([objdump, "--offloading", "library.so"], cwd=tmp_path, stdout=subprocess.DEVNULL)
    wait_states = {"v_mfma_f32_32x32x16_bf16": 12, "v_mfma_i32_16x16x64_i8": 8}

    def registers(operands):
        found = set()
        for kind, first, last, one in re.findall(r"\b([av])(?:\[(\d+):(\d+)\]|(\d+)\b)", operands):
            found |= {kind + str(r) for r in range(int(first or one), int(last or one) + 1)}
        return found

    checked, faults = [], []
    for code in sorted(tmp_path.glob("library.so.*gfx950")):
        listing = subprocess.run([objdump, "-d", code], capture_output=True, text=True, check=True).stdout
        for kernel in re.split(r"\n(?=[0-9a-f]+ <\S+>:\n)", listing)[1:]:
            if not ("MfmaGemm" in kernel[:200] and any(name in kernel for name in wait_states)):
                continue
            base, name = re.match(r"([0-9a-f]+) <(\S+)>:", kernel).groups()
            checked.append(name)
            text, at, branches = [], {}, {}
            for line in kernel.split("\n")[1:]:
                instruction, _, rest = line.partition("//")
                if not rest:
                    continue
                at[int(rest.split(":")[0], 16)] = len(text)
                if re.match(r"\s*s_c?branch", instruction):
                    branches[len(text)] = int(base, 16) + int(re.search(r"<\S+?(?:\+0x([0-9a-f]+))?>", rest).group(1) or "0", 16)
                text.append(instruction.strip())
            before = [[i - 1] if i and not text[i - 1].startswith(("s_branch", "s_endpgm")) else [] for i in range(len(text))]
            for i, target in branches.items():
                before[at[target]].append(i)
            mnemonic = [t.split(" ")[0] for t in text]
            operands = [t.partition(" ")[2].split(", ") for t in text]
            touched = [registers(t.partition(" ")[2]) for t in text]
            # (Comparisons and the like name a scalar register first; stores and loads to LDS write none.)
            written = [registers(o[0]) | (registers(o[1]) if "swap" in m and len(o) > 1 else set())
                       if m.startswith(("v_", "ds_read", "global_load", "buffer_load")) else set()
                       for m, o in zip(mnemonic, operands)]

            def close_in_front(i, states, hit):
                """Instructions less than `states` wait states in front of the i-th that `hit` says yes to."""
                ways, nearest = [(j, 0) for j in before[i]], {}
                while ways:
                    j, waited = ways.pop()
                    if waited >= states or nearest.get(j, states) <= waited:
                        continue
                    nearest[j] = waited
                    if hit(j, waited):
                        yield j
                        continue
                    waited += int(operands[j][0], 0) + 1 if mnemonic[j] == "s_nop" else 1
                    ways += [(k, waited) for k in before[j]]

            for i in range(len(text)):
                if mnemonic[i] in wait_states:
                    read = set().union(*(registers(o) for o in operands[i][1:]))
                    faults += [(name, text[j], text[i]) for j in close_in_front(
                        i, 2, lambda j, _: mnemonic[j].startswith("v_") and not mnemonic[j].startswith("v_mfma") and
                        written[j] & read)]
                elif touched[i] and not mnemonic[i].startswith("v_mfma"):
                    faults += [(name, text[j], text[i]) for j in close_in_front(
                        i, 12, lambda j, waited: waited < wait_states.get(mnemonic[j], 0) and written[j] & touched[i])]
    assert len(checked) >= 6 and any("F32Traits" in name for name in checked), checked
    assert not faults, faults[:8]


@pytest.fixture(scope="module")
def runtime_model(tmp_path_factory):
    """tests/cpp/runtime_model_test.cc: the library on a model of the HIP runtime."""
    from ruy_amd import _structs as S
    from ruy_amd import build
    exe = str(tmp_path_factory.mktemp("runtime_model") / "runtime_model_test")
    here = os.path.join(ROOT, "ruy_amd")
    rocm = os.path.dirname(os.path.dirname(build.HIPCC))
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-rdynamic", "-D__HIP_PLATFORM_AMD__",
                           "-I" + os.path.join(rocm, "include"), "-I" + os.path.join(ROOT, "include"),
                           "-I" + build.CSRC, os.path.join(ROOT, "tests", "cpp", "runtime_model_test.cc"),
                           "-L" + here, "-lruy_amd", "-Wl,-rpath," + here,
                           "-Wl,-rpath-link," + os.path.join(rocm, "lib"), "-o", exe])

    def run(what):
        result = subprocess.run([exe, what], capture_output=True, text=True)
        assert result.returncode == 0 and "all passed" in result.stdout, result.stdout + result.stderr

    def kernels():
        return subprocess.check_output([exe, "kernels"], text=True).split()

    def routes(calls):
        """What each call launches: (type tuple, M, K, N, orders) and options."""
        lines = []
        for types, M, K, N, orders, *rest in calls:
            o = dict({"pad": 0, "zero_points": True, "cached": False, "misalign": 0, "tile": (0, 0)}, **(rest[0] if rest else {}))
            zero = (3, 5) if o["zero_points"] and types[0] in (S.U8, S.I8) and types[1] in (S.U8, S.I8) else \
                tuple(128 if t == S.U8 else 0 for t in types[:2])
            lines.append("ordinary %d %d %d %d %d %d %d %d %d" % (types[0], types[1], types[3], M, K, N, *orders) +
                         " %d" % o["pad"] * 3 + " %d %d %d 0 %d %d %d" % (*zero, o["cached"], o["misalign"], *o["tile"]))
        answers = subprocess.run([exe, "routes"], input="\n".join(lines) + "\n", capture_output=True, text=True,
                                 check=True).stdout.splitlines()
        assert len(answers) == len(calls) and all(a.startswith("0 ") for a in answers)
        return [a.split()[2:] for a in answers]
    run.kernels, run.routes = kernels, routes
    return run


def test_a_failed_upload_leaves_no_cache_entry(runtime_model):
    """Whichever of a call's uploads cannot be launched, no entry packed from
    memory that was never written stays in the prepacked cache (every type)."""
    runtime_model("failed_upload")


def test_page_locked_sources_are_read_in_stream_order(runtime_model):
    """... at any alignment and size, and without a byte beyond their page."""
    runtime_model("page_locked_sources")


def test_page_locked_destinations_come_back_the_shorter_way(runtime_model):
    runtime_model("page_locked_destinations")


def test_waves_to_a_group_of_the_streaming_kernel(runtime_model):
    runtime_model("skinny_shapes")


def test_kernel_timing_leaves_the_upload_out(runtime_model):
    runtime_model("timing")


def test_one_ordinary_call_is_enough_for_a_capture(runtime_model):
    """... whatever forms the sums then, and a refused call records nothing."""
    runtime_model("capture")


def test_rows_read_where_they_lie_need_no_scratch_memory(runtime_model):
    """... under capture before any ordinary call, without allocation, and in ordinary calls."""
    runtime_model("raw_rows")


def test_calls_take_turns_with_the_pieces_of_their_scratch_memory(runtime_model):
    runtime_model("scratch_in_turns")


def test_scratch_memory_for_turns_that_cannot_be_had_is_not_asked_for_again(runtime_model):
    runtime_model("scratch_in_turns_refused")


def test_scratch_memory_in_turns_does_not_end_another_threads_recording(runtime_model):
    runtime_model("scratch_in_turns_beside_a_capture")


def test_sums_left_to_the_product_take_no_scratch_memory(runtime_model):
    runtime_model("scratch_blocks")


def test_products_the_staged_form_of_the_smallest_tile_takes(runtime_model):
    runtime_model("staged_rule")


def test_every_small_tile_kernel_is_chosen_for_a_product_that_the_gpu_tests_run(runtime_model):
    """... and the library holds no other."""
    import cases
    calls = []
    for types in cases.SMALL_TILE_TYPES:
        calls += [(types,) + p for p in cases.small_tile_problems(types)]
    launched = {kernel for route in runtime_model.routes(calls) for kernel in route if "SmallGemmKernel" in kernel}
    built = {kernel for kernel in runtime_model.kernels() if "SmallGemmKernel" in kernel}
    assert built == launched, sorted(built ^ launched)


def test_small_tiles_end_at_whole_numbers_of_tiles_to_a_cu(runtime_model):
    """A grid of a few 32x32 tiles more than three to a CU takes as long as one of
    four to a CU: 8-bit rows run where those do, from 769 tiles on."""
    from ruy_amd import _structs as S
    i8 = (S.I8, S.I8, S.I32, S.I8)
    other, small, wide = "MfmaGemmKernel", "SmallGemmKernel.*Li32ELi64ELi4E", "SmallGemmKernel.*Li64ELi64ELi8E"
    for rows, cols, ranges in [
            (768, 1024, {1024: small, 1085: small, 129: small, 257: small, 1505: small}),
            (769, 1000, {1024: other, 704: other, 1088: other, 191: small, 193: other, 257: other, 959: other, 961: small,
                         1299: small, 1301: wide, 1505: wide, 1699: wide, 1701: other}),
            (64, 12544, {1024: other, 147: small, 190: small, 250: other}),
            (1024, 1024, {1024: other, 704: other, 147: small, 190: small, 250: other, 961: small, 1505: wide})]:
        calls = [(i8, rows, depth, cols, (1, 0, 0)) for depth in ranges]
        for (_, _, depth, _, _), route in zip(calls, runtime_model.routes(calls)):
            assert re.search(ranges[depth], route[-1]), (rows, depth, cols, route)


def test_products_that_the_larger_tiles_do_faster_stay_there(runtime_model):
    """Products measured on both: (types, M, K, N, orders, padding, small tiles)."""
    from ruy_amd import _structs as S
    f32, i8i16, i16i8 = (S.F32,) * 4, (S.I8, S.I16, S.I32, S.I16), (S.I16, S.I8, S.I32, S.I16)
    i8 = (S.I8, S.I8, S.I32, S.I8)
    measured = [
        # Weights that come from HBM.
        (f32, 4096, 4096, 32, (1, 0, 0), 0, False), (f32, 8192, 2048, 64, (1, 0, 0), 0, False),      # 27.4 32.2, 27.7 31.0 us
        (f32, 8192, 4096, 96, (1, 0, 0), 0, False), (f32, 8192, 2048, 32, (1, 0, 0), 0, True),       # 69.4 77.1, 26.7 20.9
        (i8i16, 4096, 8192, 32, (1, 0, 0), 0, False), (i8i16, 8192, 4096, 64, (1, 0, 0), 0, False),  # 17.4 20.3, 17.4 19.2
        (i8i16, 8192, 4096, 32, (1, 0, 0), 0, True), (i8i16, 4096, 4096, 64, (1, 0, 0), 0, True),    # 16.1 13.9, 14.5 12.2
        (i8, 2048, 8192, 32, (1, 0, 0), 0, False), (i8, 2048, 8192, 64, (1, 1, 0), 0, False),        # 11.5 13.2, 15.1 16.7
        (i8, 8192, 8192, 32, (1, 0, 0), 0, True), (i8, 4096, 8192, 48, (1, 0, 0), 0, True),          # 18.6 16.8, 13.7 13.1
        # Operands that the caches hold.
        (f32, 2176, 288, 1520, (1, 1, 1), 0, False), (f32, 2174, 176, 1652, (1, 1, 0), 1, False),    # 28.0 33.1, 24.7 28.1 us
        (f32, 2232, 1708, 1352, (1, 0, 0), 0, False), (f32, 2048, 176, 1424, (1, 1, 0), 0, False),   # 106 116, 22.5 24.4
        (f32, 762, 28, 3856, (1, 1, 0), 0, True), (f32, 860, 2832, 1686, (1, 0, 0), 0, False),       # 15.6 11.5, 71.1 80.4
        (i8i16, 448, 3764, 2816, (1, 0, 0), 1, False), (i16i8, 1112, 1888, 1536, (0, 0, 1), 0, False),  # 37.7 53.1, 24.6 31.0
        (i8i16, 3312, 7112, 379, (0, 0, 0), 0, False), (i16i8, 3729, 3733, 390, (1, 0, 0), 1, False),   # 69.5 83.5, 50.5 59.7
        (i8i16, 191, 2624, 5940, (1, 1, 1), 0, True), (i16i8, 351, 2016, 4218, (1, 0, 0), 0, True)]     # 1.49 and 1.18 times
    calls = [(types, M, K, N, orders, {"pad": pad}) for types, M, K, N, orders, pad, _ in measured]
    for (*call, small), route in zip(measured, runtime_model.routes(calls)):
        assert ("SmallGemmKernel" in route[-1]) == small, (call, route)


def test_fp32_products_that_the_small_tiles_do_faster_run_there(runtime_model):
    """Narrow and shallow products near the line to the tiles on bf16 parts, measured on
    both, us: small tiles, larger ones."""
    from ruy_amd import _structs as S
    calls = [((S.F32,) * 4, M, K, N, orders) for M, K, N, orders in [
        (205, 2112, 352, (1, 0, 0)), (190, 926, 5936, (1, 0, 0)),      # 13.2 15.4, 29.8 33.9
        (124, 2067, 288, (1, 0, 0)), (212, 1902, 128, (1, 0, 0)),      # 13.0 15.1, 12.5 14.9
        (1035, 2288, 81, (1, 0, 0)), (488, 1552, 2336, (1, 0, 0)),     # 14.5 16.2, 41.7 45.6
        (194, 2208, 1300, (1, 1, 0)), (112, 2812, 1280, (0, 0, 1)),    # 27.5 35.4, 19.2 20.9
        (1643, 112, 1502, (1, 1, 1)), (1088, 112, 2145, (0, 0, 1))]]   # 15.4 18.8, 15.4 17.4
    for call, route in zip(calls, runtime_model.routes(calls)):
        assert "SmallGemmKernel" in route[-1], (call, route)


def test_products_of_the_staged_tests_run_on_every_staged_kernel(runtime_model):
    """Both rings, both alignments, with sums and without, each beside rows of the
    other operand that come from the cache."""
    import cases
    raw, cached = set(), set()
    for depth in cases.STAGED_DEPTHS:
        calls = [(types, rows, depth, cols, (1, 0, depth % 2),
                  {"pad": pad, "cached": from_cache, "misalign": misalign, "zero_points": zero_points, "tile": (64, 64)})
                 for types in cases.STAGED_TYPES for rows, cols, pad, from_cache in cases.STAGED_SHAPES
                 for misalign in (0, 1) for zero_points in (False, True)]
        for call, route in zip(calls, runtime_model.routes(calls)):
            (cached if call[-1]["cached"] else raw).update(k for k in route if "GemmKernel" in k)
    staged = re.compile(r"MfmaGemmKernel\w+Int8Traits\w*Lb0ELi[12]EEEv")
    built = {k for k in runtime_model.kernels() if staged.search(k)}
    assert len(built) == 8
    assert built <= raw, sorted(built - raw)
    assert built <= cached, sorted(built - cached)


def test_products_of_the_pack_tests_are_packed(runtime_model):
    import cases
    from ruy_amd import _structs as S
    for depth in cases.PACK_DEPTHS:
        calls = [((S.U8, S.U8, S.I32, S.U8), rows, depth, cols, orders, {"pad": depth % 4 == 1, "tile": (128, 128)})
                 for rows, cols in cases.PACK_SHAPES for orders in cases.PACK_ORDERS]
        for call, route in zip(calls, runtime_model.routes(calls)):
            assert "PackKernel" in route[0], (call, route)


def test_fp32_grids_of_the_ring_tests_run_on_two_stages(runtime_model):
    import cases
    from ruy_amd import _structs as S
    for tile, rows, cols in cases.F32_SHALLOW_RINGS:
        for depth in (5, 1111):
            calls = [((S.F32,) * 4, rows, depth, cols, (1, 0, 0), {"pad": 1, "misalign": 4, "tile": tile})]
            form = "MfmaGemmKernelINS_12_GLOBAL__N_19F32TraitsELi%dELi%dELi128ELi2E" % (tile[0] // 64, tile[1] // 64)
            assert [form in kernel for kernel in runtime_model.routes(calls)[0]] == [True]


@pytest.mark.skipif(not os.path.isdir(os.path.join(REFERENCE, "example")),
                    reason="reference tree not present")
@pytest.mark.parametrize("std", ["c++14", "c++17"])
def test_reference_examples_compile_against_our_headers(std, tmp_path):
    """The reference's two example programs must build unchanged: that is the
    source-level drop-in claim. (Running them needs a GPU; the same cases are
    executed by tests/cpp/api_test.cc.)"""
    for name in ("example.cc", "parametrized_example.cc"):
        obj = str(tmp_path / (name + ".o"))
        subprocess.check_call(["g++", "-std=" + std, "-I" + os.path.join(ROOT, "include"), "-c",
                               os.path.join(REFERENCE, "example", name), "-o", obj])
        exe = str(tmp_path / name.replace(".cc", ""))
        subprocess.check_call(["g++", obj, "-L" + os.path.join(ROOT, "ruy_amd"), "-lruy_amd", "-o", exe])


def test_python_mirror_defaults():
    """ruy/mul_params_test.cc:26-72 and ruy/matrix_test.cc on the Python mirror."""
    from ruy_amd import _structs as S
    from ruy_amd import api
    p = api.MulParams(S.I32, S.I8)
    assert p.bias is None
    assert p.multiplier_fixedpoint() == 0 and p.multiplier_exponent() == 0
    assert p.multiplier_fixedpoint_perchannel() is None
    assert (p.clamp_min, p.clamp_max) == (-128, 127)
    assert p.channel_dimension == api.ChannelDimension.kRow
    assert p.perchannel_buffers_capacity_rounding() == 1
    p.set_multiplier_fixedpoint(123)
    p.set_multiplier_exponent(4)
    p.set_perchannel_buffers_capacity_rounding(8)
    assert (p.multiplier_fixedpoint(), p.multiplier_exponent()) == (123, 4)
    assert p.perchannel_buffers_capacity_rounding() == 8
    p.set_multiplier_fixedpoint(0)
    p.set_multiplier_exponent(0)
    p.set_multiplier_fixedpoint_perchannel([1])
    p.set_multiplier_exponent_perchannel([1])
    assert p.multiplier_fixedpoint() == 0 and p.multiplier_fixedpoint_perchannel() == [1]
    f = api.MulParams(S.F32, S.F32)
    assert f.clamp_min == float("-inf") and f.clamp_max == float("inf")
    with pytest.raises(ValueError):
        api.MulParams(S.F32, S.I8)
    with pytest.raises(ValueError):
        api.MulParams(S.I32, S.F32)
    lay = api.make_simple_layout(3, 5, api.Order.kRowMajor)
    assert lay.stride == 5 and api.offset(lay, 2, 1) == 11
    lay = api.make_simple_layout(3, 5, api.Order.kColMajor)
    assert lay.stride == 3 and api.offset(lay, 2, 1) == 5
    m = api.Matrix(S.U8)
    assert m.zero_point == 0 and m.cache_policy == api.CachePolicy.kNeverCache


def test_context_creation_fails_loudly_without_a_gpu():
    import torch
    if torch.cuda.is_available():
        pytest.skip("a GPU is present")
    from ruy_amd import api
    with pytest.raises(api.RuyAmdError):
        api.Context()


def test_product_code_never_touches_the_checker():
    """The CPU checker under oracle/ is test infrastructure: nothing in the
    package or in the public headers may include, import, load or name it, and
    the package has no CPU fallback to route through."""
    roots = [os.path.join(ROOT, "ruy_amd"), os.path.join(ROOT, "include")]
    pattern = re.compile(r"oracle|libstock_ruy|libruy_oracle|_ref/")
    offenders = []
    for root in roots:
        for dirpath, dirnames, filenames in os.walk(root):
            dirnames[:] = [d for d in dirnames if d not in ("__pycache__", "_obj")]
            for name in filenames:
                if not name.endswith((".py", ".h", ".cc", ".hip")):
                    continue
                path = os.path.join(dirpath, name)
                with open(path, encoding="utf-8") as f:
                    for number, line in enumerate(f, 1):
                        if pattern.search(line):
                            offenders.append("%s:%d: %s" % (os.path.relpath(path, ROOT), number, line.strip()))
    assert not offenders, "\n".join(offenders)


def test_tile_choice_of_the_timing_model():
    """The tile the tiled kernels run a shape on is host arithmetic (a timing
    model fitted to measurements, ruyamd_diag_tile_for): the benchmark
    configurations that rely on the smallest tile (the batched launch of the
    small ones, which run on the small tiles one by one; the int16 operand read
    in place) get it, the 8192^3 product gets
    the 256 x 256 tile, few tiles with a long depth split it over workgroups,
    and the choice splits the depth on no other tile but the 256 x 256 one of
    the int8 kernel. Arguments that make no sense are refused."""
    from ruy_amd import api
    assert api.tile_for(0, 256, 256, 256) == (64, 64, 1)        # C1
    assert api.tile_for(2, 1024, 1024, 1024) == (64, 64, 1)     # C2
    assert api.tile_for(0, 1024, 1024, 196) == (64, 64, 1)      # C3
    assert api.tile_for(1, 2048, 2048, 512) == (64, 64, 1)      # C4: 64 rows x 128 plane columns
    assert api.tile_for(0, 8192, 8192, 8192) == (256, 256, 1)   # the headline product
    assert api.tile_for(0, 4096, 4096, 4096) == (256, 256, 1)   # exactly one round of large tiles
    rows, cols, parts = api.tile_for(0, 128, 65536, 128)
    assert (rows, cols) == (64, 64) and parts == 32
    # Few 256x256 tiles with a very long depth: that tile, its depth dealt to 2, 4 or 8 workgroups.
    assert api.tile_for(0, 2048, 16384, 2048) == (256, 256, 4)
    assert api.tile_for(0, 2048, 32768, 1024) == (256, 256, 8)
    assert api.tile_for(0, 2048, 8192, 2048) == (128, 128, 1)   # not worth it at this depth
    assert api.tile_for(0, 1024, 32768, 1024) == (256, 256, 8)  # ... rather than 256 of the 64x64 tiles
    assert api.tile_for(0, 1024, 16384, 1024) == (64, 64, 1)
    assert api.tile_for(0, 2560, 8192, 2560) == (256, 256, 2)
    rows, cols, parts = api.tile_for(2, 64, 32768, 64)
    assert (rows, cols) == (64, 64) and parts > 1
    for kind in (0, 1, 2):
        for m, k, n in [(300, 300, 300), (1536, 512, 4096), (2048, 2048, 2048), (5000, 5000, 5000), (16384, 16384, 256)]:
            rows, cols, parts = api.tile_for(kind, m, k, n)
            # (int8 x int16: a tile's plane columns are half as many destination columns)
            tiles = ((256, 128), (128, 64), (64, 64)) if kind == 1 else \
                ((256, 256), (128, 128), (128, 64), (64, 128), (64, 64))
            assert (rows, cols) in tiles, (kind, m, k, n)
            # Only the smallest tile splits the depth, and the 256x256 tile of the int8 kernel.
            assert parts == 1 or (rows, cols) == (64, 64) or (kind == 0 and (rows, cols) == (256, 256)), \
                (kind, m, k, n)
    # Fewer compute units: a grid that fills 256 CUs once is four rounds on 64 and stays on the large tile.
    assert api.tile_for(0, 4096, 4096, 4096, compute_units=64) == (256, 256, 1)
    for bad in [(3, 64, 64, 64), (0, 0, 64, 64), (0, 64, -1, 64), (0, 64, 64, 0)]:
        with pytest.raises(ValueError):
            api.tile_for(*bad)
    with pytest.raises(ValueError):
        api.tile_for(0, 64, 64, 64, compute_units=0)



def test_the_native_call_path_gathers_what_to_struct_does():
    """api.mul's native path (csrc/python/native.cc) hands ruyamd_mul the same
    structs as the Python conversion, and leaves what it does not handle to it."""
    import ctypes as C
    import numpy as np
    import torch
    from ruy_amd import _structs as S
    from ruy_amd import api
    from ruy_amd._capi import lib, native
    seen = []
    proto = C.CFUNCTYPE(C.c_int, C.c_void_p, C.POINTER(S.Mat), C.POINTER(S.Mat), C.POINTER(S.MulParamsStruct),
                        C.POINTER(S.Mat))

    def fields(struct):  # (without the padding behind the last one)
        return bytes(struct)[:type(struct).reserved.offset + 1]

    def capture(ctx, lhs, rhs, params, dst):
        seen.append((ctx,) + tuple(fields(x.contents) for x in (lhs, rhs, params, dst)))
        return 7

    callback = proto(capture)
    kinds = (api.Matrix, api.Layout, api.MulParams)
    native.bind(C.cast(callback, C.c_void_p).value, *kinds)
    try:
        buffers = [np.zeros(64, np.int8), torch.zeros(64, dtype=torch.int8), 1 << 40, None]
        for i, data in enumerate(buffers):
            lhs = api.Matrix(S.I8, data, api.Layout(3 + i, 5, 2 ** 31 - 1 - i, 1), -7 - i, 3)
            rhs = api.Matrix(S.U8, buffers[i - 1], api.Layout(5, 4, 5, 0), 255, 0)
            dst = api.Matrix(S.I16, buffers[1], api.Layout(3 + i, 4, 9, 0), 2 ** 32 + 3)
            params = api.MulParams(S.I32, S.I16)
            params.set_bias(data)
            params.set_clamp_min(-5)
            params.set_clamp_max(np.float64(77.5))
            params.set_channel_dimension(i % 2)
            params.set_perchannel_buffers_capacity_rounding(8)
            if i % 2:
                params.set_multiplier_fixedpoint(-(2 ** 31) + i)
                params.set_multiplier_exponent(-9)
            else:
                params.set_multiplier_fixedpoint_perchannel(buffers[0])
                params.set_multiplier_exponent_perchannel(buffers[1])
            assert native.mul(lhs, rhs, params, 1234, dst) == 7
            want = tuple(fields(x.to_struct()) for x in (lhs, rhs, params, dst))
            assert seen.pop() == (1234,) + want
        # Left to the Python path: other types, values that need converting, mismatched types.
        class Other(api.Matrix):
            pass
        assert native.mul(Other(S.I8), rhs, params, 1, dst) is None
        lhs.zero_point = 2.0
        assert native.mul(lhs, rhs, params, 1, dst) is None
        lhs.zero_point = 2
        lhs.data = object()
        assert native.mul(lhs, rhs, params, 1, dst) is None
        lhs.data = None
        dst.dtype = S.I8
        assert native.mul(lhs, rhs, params, 1, dst) is None
        assert not seen
    finally:
        native.bind(C.cast(lib.ruyamd_mul, C.c_void_p).value, *kinds)


def test_the_native_call_path_holds_what_it_asks():
    """A buffer that takes itself out of its matrix when asked for its address,
    and a bound that takes the other one away: both are still there when they are
    asked the next thing."""
    from ruy_amd import _structs as S
    from ruy_amd import api
    from ruy_amd._capi import native
    events = []

    class Tracked:
        def __init__(self, name):
            self.name = name

        def __del__(self):
            events.append(self.name + " gone")

    class Buffer(Tracked):
        def data_ptr(self):
            rhs.data = None
            raise AttributeError("data_ptr")

        @property
        def ctypes(self):
            events.append("buffer asked")
            raise AttributeError("ctypes")

    class Bound(Tracked):
        def __float__(self):
            events.append(self.name + " asked")
            params.clamp_max = 1.0
            return 0.0

    layout = api.Layout(4, 4, 4, 0)
    lhs, rhs, dst = api.Matrix(S.I8, 0, layout), api.Matrix(S.I8, Buffer("buffer"), layout), api.Matrix(S.I8, 0, layout)
    params = api.MulParams(S.I32, S.I8)
    params.clamp_min, params.clamp_max = Bound("lower"), Bound("upper")
    assert native.mul(lhs, rhs, params, 0, dst) is None
    assert events == ["lower asked", "upper asked", "upper gone", "buffer asked", "buffer gone"]


def test_the_package_works_without_its_native_call_path():
    """Another interpreter than the one it was built for, or one without its
    headers: the mirror's own conversion makes the same calls."""
    code = """if 1:
        import sys, warnings
        sys.modules["ruy_amd._native"] = None  # importing it raises ImportError
        with warnings.catch_warnings(record=True) as caught:
            warnings.simplefilter("always")
            from ruy_amd import _structs as S, api
        assert any("_native" in str(w.message) for w in caught), caught
        calls = []
        class Lib:
            def ruyamd_mul(self, ctx, l, r, p, d):
                calls.append((l._obj.rows, r._obj.cols, p._obj.clamp_max, d._obj.stride))
                return 0
        class Context:
            _h, _address = None, 0
            def _check(self, rc):
                assert rc == 0
        api.lib = Lib()
        make = lambda rows, cols: api.Matrix(S.I8, 4096, api.make_simple_layout(rows, cols, api.Order.kColMajor))
        api.mul(make(3, 5), make(5, 7), api.MulParams(S.I32, S.I8), Context(), make(3, 7))
        assert calls == [(3, 7, 127.0, 3)], calls
    """
    subprocess.check_call([sys.executable, "-c", code], cwd=ROOT)


def test_the_native_call_path_is_built_where_it_can_be_and_when_it_has_to(tmp_path, monkeypatch):
    from ruy_amd import build
    monkeypatch.setattr(build, "NATIVE", str(tmp_path / "_native.so"))
    paths = build.sysconfig.get_paths()
    monkeypatch.setattr(build.sysconfig, "get_paths", lambda: dict(paths, include=str(tmp_path)))
    assert build.build_native() is None and not os.path.exists(build.NATIVE)  # no Python.h there
    monkeypatch.setattr(build.sysconfig, "get_paths", lambda: paths)
    if not os.path.exists(os.path.join(paths["include"], "Python.h")):
        pytest.skip("this interpreter has no headers")
    assert build.build_native() == build.NATIVE
    built = os.stat(build.NATIVE).st_mtime_ns
    build.build_native()
    assert os.stat(build.NATIVE).st_mtime_ns == built  # up to date: left alone
    build.build_native(force=True)
    assert os.stat(build.NATIVE).st_mtime_ns > built
