"""The built code of every object that holds kernels with one hierarchy per lane, ahead of time and
at run time (hiprtc), against a fault of the compiler's register allocation: a vector register copied
at the head of a join block before `s_or_b64 exec` keeps its value only in the lanes of the branch just
left.  `-sgpr-regalloc=basic` (KERNEL_FLAGS of symboltz.build) keeps the compiler from it."""
import re
import subprocess
from concurrent.futures import ThreadPoolExecutor

from symboltz import _lib, build, models
from symboltz.multi import multi_cache_path, multi_source
from symboltz.solver import _declare, has_group, model_source

LLVM = "/opt/rocm/llvm/bin/"
COPY = re.compile(r"v_accvgpr|v_mov_b(32|64)\S* v\S+ v|scratch_")


def listing(path, tmp):
    """Disassembly with branch targets as labels, of a code object or of the bundle that holds it."""
    elf = path
    if path.read_bytes()[:4] != b"\x7fELF":
        elf = tmp / (path.stem + ".co")
        subprocess.run([LLVM + "clang-offload-bundler", "--unbundle", "--type=o", f"--input={path}",
                        "--targets=hipv4-amdgcn-amd-amdhsa--gfx950", f"--output={elf}"], check=True)
    return subprocess.run([LLVM + "llvm-objdump", "-d", "--symbolize-operands", "--no-show-raw-insn",
                           "--no-leading-addr", str(elf)], check=True, capture_output=True, text=True).stdout


def lost_copies(asm):
    """(kernels seen, [(kernel, label, first copy) of every join block whose head copies before its mask])"""
    bad, kernels = [], 0
    for part in re.split(r"\n(?=<sbz_\w+>:)", asm)[1:]:
        kernels += 1
        joins = set(re.findall(r"s_cbranch_execn?z (L\d+)", part))
        for block in re.split(r"\n(?=<L\d+>:)", part)[1:]:
            label = block[1:block.index(">")]
            head = []
            for line in block.split("\n")[1:] if label in joins else []:
                t = line.split("//")[0].strip()
                if t.startswith("s_or_b64 exec, exec"):
                    if head and all(COPY.match(h) for h in head):
                        bad.append((part[1:part.index(">")], label, head[0]))
                    break
                if re.match(r"s_cbranch|s_branch|s_endpgm|s_\w+ exec|s_\w+_saveexec", t):
                    break
                if t.startswith(("v_", "ds_", "global_", "scratch_")) and not t.startswith(("v_readlane", "v_writelane")):
                    head.append(t)
    return kernels, bad


def ahead_of_time():
    """(name, source, path in the code object cache)"""
    out = [(f"n{M.n_unknowns}", model_source(M).full_src, build.KCACHE / f"{model_source(M).full_hash}.hsaco")
           for M in build.standard_models() + build.layout_models()]
    for i, fams in enumerate(build.standard_multis()):
        for rows in (False, True):
            src = multi_source(fams, rows_kernel=rows)
            out.append((f"mixed{i}{'rows' if rows else ''}", src, multi_cache_path(src)))
    return [o for o in out if has_group(o[1])]


def test_ahead_of_time_objects(tmp_path):
    work = ahead_of_time()
    assert len(work) >= 9

    def scan(w):
        name, src, path = w
        if not path.exists():
            path = build.compile_code_object(src, tmp_path / f"{name}.hsaco")
        return name, *lost_copies(listing(path, tmp_path))
    with ThreadPoolExecutor(6) as ex:
        for name, kernels, bad in ex.map(scan, work):
            assert kernels >= (1 if name.startswith("mixed") else 8) and not bad, (name, kernels, bad)


# the shortest lanes, the last with the kept factors and the look-ahead interval (12 slots), the first
# without, the longest, and seven hierarchies without massless neutrinos
RUN_TIME = [dict(lmax=3, h=False), dict(lmax=5), dict(lmax=11), dict(lmax=12),
            dict(lmax_g=17, lmax_nu=4, lmax_h=3, nx=2), dict(lmax=6, nu=False, nx=5)]


def test_run_time_objects(tmp_path):
    L = _lib.lib()
    _declare(L)
    srcs = [model_source(models.LCDM(**kw)).full_src for kw in RUN_TIME]   # emission is not for threads

    def scan(i):
        path = tmp_path / f"{i}.co"
        assert has_group(srcs[i])
        assert L.sbz_compile(srcs[i].encode(), str(path).encode()) == 0
        return RUN_TIME[i], *lost_copies(listing(path, tmp_path))
    with ThreadPoolExecutor(6) as ex:
        for kw, kernels, bad in ex.map(scan, range(len(RUN_TIME))):
            assert kernels >= 8 and not bad, (kw, kernels, bad)


def test_without_its_flag_the_fault_is_there_and_found(tmp_path):
    src, out = tmp_path / "m.hip", tmp_path / "m.hsaco"
    src.write_text(model_source(models.LCDM(lmax=6)).full_src)
    assert build.KERNEL_FLAGS[-2:] == ["-mllvm", "-sgpr-regalloc=basic"]
    subprocess.run(["hipcc", "--genco"] + build.KERNEL_FLAGS[:-2] + [str(src), "-o", str(out)], check=True,
                   stderr=subprocess.DEVNULL)
    kernels, bad = lost_copies(listing(out, tmp_path))
    assert kernels >= 8 and {k for k, _, _ in bad} & {"sbz_wave2h_kernel", "sbz_group_save_kernel"}
