"""The built GPU code held to rules of the instruction set that inline assembly can break
without an error: what the compiler's hazard pass sees to by itself for its own instructions, it
cannot see inside an asm statement."""
import os
import re
import struct
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "glm.c_amd", "libgmoe.so")
OBJDUMP = os.path.join(os.environ.get("ROCM", "/opt/rocm"), "llvm", "bin", "llvm-objdump")
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def code_objects():
    """The gfx950 code objects of libgmoe.so (one per source file), from its offload bundles."""
    data = open(LIB, "rb").read()
    found, at = [], data.find(MAGIC)
    while at >= 0:
        (n,) = struct.unpack_from("<Q", data, at + len(MAGIC))
        p = at + len(MAGIC) + 8
        if n < 16:  # (the magic's own text elsewhere is not a bundle)
            for _ in range(n):
                off, size, idlen = struct.unpack_from("<QQQ", data, p)
                name = data[p + 24:p + 24 + idlen]
                p += 24 + idlen
                if b"gfx950" in name and size:
                    found.append(data[at + off:at + off + size])
        at = data.find(MAGIC, at + 1)
    return found


@pytest.fixture(scope="module")
def listing(tmp_path_factory):
    """[instruction lines] of every code object."""
    objs = code_objects()
    assert objs, "no gfx950 code in libgmoe.so"
    lines = []
    for i, blob in enumerate(objs):
        path = tmp_path_factory.mktemp("co") / f"{i}.co"
        path.write_bytes(blob)
        out = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", "--no-leading-addr", str(path)], check=True,
                             capture_output=True, text=True).stdout
        lines += [re.sub(r"\s*//.*", "", s).strip() for s in out.splitlines() if s.startswith((" ", "\t"))]
    return lines


def test_m0_write_has_a_wait_state_before_a_dma_reads_it(listing):
    """An LDS DMA takes its destination from m0, and a scalar write of m0 needs one wait state (any
    other instruction) before it; the compiler puts an s_nop there where it has nothing else."""
    dma = [i for i, s in enumerate(listing) if re.match(r"(global|buffer)_load_(lds_|.*\blds$)", s)]
    assert len(dma) > 100, "the listing's DMAs were not recognised"
    bad = [f"{listing[i - 1]} / {listing[i]}" for i in dma if re.match(r"s_\w+ m0,", listing[i - 1])]
    assert not bad, f"{len(bad)} of {len(dma)} DMAs read m0 right after its write, e.g. {bad[0]}"


def sgprs(text):
    """The scalar registers that an operand list names."""
    regs = {int(m) for m in re.findall(r"\bs(\d+)\b", text)}
    for a, b in re.findall(r"\bs\[(\d+):(\d+)\]", text):
        regs |= set(range(int(a), int(b) + 1))
    return regs


def test_no_vector_write_of_a_scalar_address_right_before_its_load(listing):
    """A scalar register that a vector instruction wrote (v_readfirstlane) needs five wait states
    before a memory instruction takes it as its address."""
    bad = []
    for i, s in enumerate(listing):
        used = sgprs(s) if re.match(r"(global|buffer)_", s) else ()
        states, j = 0, i - 1
        while used and states < 5 and j >= 0:
            op, _, rest = listing[j].partition(" ")
            if op.startswith("v_") and sgprs(rest.split(",")[0]) & used:
                bad.append(f"{listing[j]} / {s}")
            states += int(rest) + 1 if op == "s_nop" else 1
            j -= 1
    assert not bad, f"{len(bad)} loads, e.g. {bad[0]}"


def test_no_shared_memory_read_is_under_way_at_a_barrier(listing):
    """After a barrier other waves (and their DMAs) write what a wave read before it, so its reads
    have returned by then; __builtin_amdgcn_s_barrier() neither waits for them nor keeps the
    compiler from moving them over it."""
    pending, bad = 0, 0
    for s in listing:
        wait = re.search(r"lgkmcnt\((\d+)\)", s)
        if s == "s_endpgm":
            pending = 0
        elif wait:
            pending = min(pending, int(wait[1]))
        elif s.startswith("ds_read"):
            pending += 1
        elif s.startswith("s_barrier"):
            bad += pending > 0
    assert bad == 0, f"{bad} barriers with reads of shared memory under way"


def test_batch_attention_exponential():
    """a16_exp (attn16.h) restated with its constants read from the source: 2^(x log2 e), the product
    in two parts, its rounding's error joining as 1 + r ln 2 with |r| < 2^-16. With a correctly
    rounded 2^t two roundings of half an ulp are left, of 2^t and of the result, so within 1.1 ulp of
    e^x over [-87, 6]; the instruction's own 2^t measures 1.26 over every float."""
    import numpy as np

    src = open(os.path.join(ROOT, "glm.c_amd", "csrc", "attn16.h")).read()
    L, L2, LN2 = (np.float32(v) for v in re.search(r"const float L = (\S+)f, L2 = (\S+)f, LN2 = (\S+)f;", src).groups())
    assert abs(float(L) + float(L2) - np.log2(np.e)) < 2.0 ** -48
    x = np.random.default_rng(2).uniform(-87, 6, 1 << 20).astype(np.float32)
    d = np.float64
    t = (d(x) * d(L)).astype(np.float32)
    r = (d(x) * d(L2) + d((d(x) * d(L) - d(t)).astype(np.float32))).astype(np.float32)
    e = np.exp2(d(t)).astype(np.float32)
    got = (d(e) * d((d(r) * d(LN2)).astype(np.float32)) + d(e)).astype(np.float32)
    want = np.exp(d(x))
    assert (np.abs(d(got) - want) / np.spacing(want.astype(np.float32))).max() < 1.1
