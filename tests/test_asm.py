"""Properties of the gfx950 code the library ships, checked on the assembly hipcc emits for its sources (CPU only: hipcc
cross-compiles here).

- No kernel uses scratch (private segment) apart from the listed ones: the debug instantiations (int32 unit values
  written out for the tests).
- The decode product at 3-32 tokens and the prefill kernels on packed trits read global memory only through buffer resources
  that span exactly their buffers, so an out-of-range offset reads zeros and cannot fault; the q8_0 product at many tokens
  reads its weights, activations and scales so (its list tables, 4 bytes an entry, directly).
- The prefill kernels wait for their DMAs by count: the counts they wait with are the DMAs they issue.
- No kernel writes through the scalar data cache.
"""
import os
import re
import shutil
import subprocess
from concurrent.futures import ThreadPoolExecutor

import pytest

from kindi_amd import build

pytestmark = pytest.mark.skipif(not os.path.exists(build.HIPCC) and shutil.which("hipcc") is None,
                                reason="hipcc is not installed")


def _asm(src, tmp):
    out = os.path.join(tmp, src.replace(".hip", ".s"))
    cmd = [build.HIPCC] + build.FLAGS + ["-S", "--cuda-device-only", os.path.join(build.CSRC, src), "-o", out]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    return open(out).read()


@pytest.fixture(scope="module")
def asm(tmp_path_factory):
    tmp = str(tmp_path_factory.mktemp("asm"))
    with ThreadPoolExecutor(min(8, len(build.SOURCES))) as ex:
        texts = list(ex.map(lambda s: _asm(s, tmp), build.SOURCES))
    return dict(zip(build.SOURCES, texts))


def _kernels(text):
    """{mangled name: (body lines, metadata block)} of every kernel in one assembly file"""
    out = {}
    lines = text.split("\n")
    for i, l in enumerate(lines):
        m = re.match(r"^(_Z\S+|k_\w+):\s", l + " ")
        if m and i + 1 < len(lines):
            name = m.group(1)
            body = []
            for l2 in lines[i + 1:]:
                if l2.startswith((".Lfunc_end", "\t.section")):         # past every s_endpgm: a kernel may return early
                    break
                body.append(l2.strip())
            out[name] = [body, None]
    for blk in text.split("  - .agpr_count")[1:]:
        nm = re.search(r"\.name:\s+(\S+)", blk)
        sym = re.search(r"\.symbol:\s+(\S+)\.kd", blk)
        if sym and sym.group(1) in out:
            out[sym.group(1)][1] = blk
        elif nm:
            out.setdefault(nm.group(1), [[], None])[1] = blk
    return out


SCRATCH_OK = {"k_gemv_flat1<0, 1, true, false>", "k_gemv_pair<true>", "k_q8_mma<false, true, false, true>",
              "k_q8_mma<true, true, false, true>", "k_q8_mma<true, true, false, false>", "k_tern_gemm8<true>", "k_gemv_m16<true, 2, true, true>"}


def _demangle(names):
    tool = shutil.which("c++filt") or shutil.which("llvm-cxxfilt")
    if tool is None:
        return {n: n for n in names}
    r = subprocess.run([tool], input="\n".join(names), capture_output=True, text=True)
    return dict(zip(names, [l.split("(")[0].replace("void ", "") for l in r.stdout.split("\n")]))


def test_no_kernel_uses_scratch(asm):
    seen, used = 0, set()
    for src, text in asm.items():
        ks = {n: m for n, (_, m) in _kernels(text).items() if m is not None}
        dm = _demangle(list(ks))
        for name, meta in ks.items():
            seen += 1
            priv = int(re.search(r"\.private_segment_fixed_size:\s+(\d+)", meta).group(1))
            spill = int(re.search(r"\.vgpr_spill_count:\s+(\d+)", meta).group(1))
            if priv or spill:
                used.add(dm[name])
    assert seen >= 20
    assert used <= SCRATCH_OK, sorted(used - SCRATCH_OK)


def _ops(body):
    return [l.split()[0] for l in body if l and not l.startswith((".", ";")) and not l.endswith(":")]


@pytest.mark.parametrize("src,pat", [("kt_mma.hip", "k_gemv_m16"), ("kt_prefill.hip", "k_tern_gemm_w"), ("kt_prompt.hip", "k_tern_gemm_ks")])
def test_reads_through_buffer_resources(asm, src, pat):
    ks = {n: b for n, (b, _) in _kernels(asm[src]).items() if pat in n and b}
    assert ks, pat
    for name, body in ks.items():
        ops = _ops(body)
        flat = [o for o in ops if o.startswith(("global_load", "flat_load", "global_atomic", "flat_atomic"))]
        assert not flat, (name, flat[:5])
        assert any(o.startswith("buffer_load") for o in ops), name


def test_q8_gemm_reads(asm):
    """k_q8_gemm: dense, everything through buffer resources; grouped, the list tables (single words) beside them"""
    ks = {n: b for n, (b, _) in _kernels(asm["kt_q8gemm.hip"]).items() if "k_q8_gemm" in n and b}
    assert len(ks) == 4
    for name, body in ks.items():
        ops = _ops(body)
        flat = {o for o in ops if o.startswith(("global_load", "flat_load", "global_atomic", "flat_atomic"))}
        assert flat <= ({"global_load_dword"} if "ILb1E" in name else set()), (name, flat)
        assert sum(o.startswith("buffer_load") for o in ops) > 24, name


# the DMAs a wave issues for one stage: k_tern_gemm_w<T>: T of activations, packed trits, row scales (and token scales without
# RS); k_tern_gemm_ks: 4, 1, 1 (and 1)
@pytest.mark.parametrize("src,pat,dmas,last", [("kt_prefill.hip", r"k_tern_gemm_wILi(\d)ELb(\d)ELb0E", lambda t, rs: t + 3 - rs, lambda t: 16 * t),
                                          ("kt_prompt.hip", r"k_tern_gemm_ksILi(\d)ELb(\d)ELb0E", lambda nw, rs: 7 - rs, lambda nw: 16 // nw)])
def test_dma_waits_are_counted(asm, src, pat, dmas, last):
    """loads retire in order, so a wait for all but n leaves exactly the last n in flight: n is the DMAs of one stage, each
    stage between two barriers issues that many or none, and the only other loads are the outputs' token scales at the end (RS)"""
    seen = 0
    for name, (body, _) in _kernels(asm[src]).items():
        m = re.search(pat, name)
        if not m or not body:
            continue
        seen += 1
        v, rs = int(m.group(1)), int(m.group(2))
        n = dmas(v, rs)
        lds = [i for i, l in enumerate(body) if l.startswith("buffer_load") and l.endswith(" lds")]
        other = [i for i, l in enumerate(body) if re.match(r"(buffer|global|flat|scratch)_load", l) and i not in lds]
        assert lds and len(lds) % n == 0 and len(other) == (last(v) if rs else 0), (name, len(lds), len(other), n)
        waits = {int(w) for w in re.findall(r"s_waitcnt vmcnt\((\d+)\)", "\n".join(body))}
        assert waits == {0, n} or waits == {n}, (name, waits, n)
        run = 0
        for l in body + ["s_barrier"]:
            if l.startswith(("s_barrier", "s_cbranch", "s_branch")) or l.endswith(":"):
                assert run % n == 0, (name, run, n)
                run = 0
            run += l.startswith("buffer_load") and l.endswith(" lds")
    assert seen == 4


def test_no_scalar_cache_writes(asm):
    for src, text in asm.items():
        for l in text.split("\n"):
            op = l.strip().split(" ")[0] if l.strip() else ""
            assert not op.startswith(("s_store", "s_scratch_store", "s_buffer_store", "s_atomic", "s_buffer_atomic",
                                      "s_dcache_wb")), (src, l)
