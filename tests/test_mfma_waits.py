"""The matrix products that csrc/gemm_tile.h writes in asm, in the assembly that the build's compiler makes of the kernels that use them.  The compiler does
not know what such an instruction takes, so it adds no waits around it: whatever it puts near one (a move of the sums, a copy of an operand) has to lie far
enough away by the order of the code alone.  A product of 16 x 16 x 32 (4 passes) leaves its sums to others after 8 wait states, as the compiler waits after its own, and takes
registers that another instruction wrote after 2; an instruction is one, s_nop n is n + 1."""

import re
import subprocess

import pytest

from neuronx_distributed_llama3_2_amd import _build

SUMS, OPERANDS = 8, 2


def _regs(text):
    """Registers named in operands: a5, v[8:11] -> {('a', 5), ('v', 8), ...}."""
    out = set()
    for kind, one, lo, hi in re.findall(r"\b([av])(?:(\d+)|\[(\d+):(\d+)\])", text):
        out.update((kind, r) for r in ([int(one)] if one else range(int(lo), int(hi) + 1)))
    return out


def _functions(asm):
    """{name: ([(instruction, operands)], {label: index})} of the kernels."""
    funcs, cur = {}, None
    for line in asm.splitlines():
        line = line.split(";")[0].rstrip()
        m = re.match(r"([\w.$]+):", line)
        if m:
            if not m.group(1).startswith(".L"):
                cur = funcs.setdefault(m.group(1), ([], {}))
            elif cur is not None:
                cur[1][m.group(1)] = len(cur[0])
        elif cur is not None and re.match(r"\s+[a-z]", line):
            op, _, args = line.strip().partition(" ")
            cur[0].append((op, args))
        elif line.strip().startswith(".section"):
            cur = None
    return funcs


def _close(code, labels):
    """What lies too near a product: (distance, the first instruction, the second)."""
    before = [[i - 1] if i and code[i - 1][0] not in ("s_branch", "s_endpgm", "s_setpc_b64") else [] for i in range(len(code))]
    for i, (op, args) in enumerate(code):
        if op.startswith(("s_branch", "s_cbranch")) and args.strip() in labels and labels[args.strip()] < len(code):
            before[labels[args.strip()]].append(i)
    split = lambda i: [_regs(a) for a in re.split(r",\s*(?![^\[]*\])", code[i][1])]
    mfma = lambda i: code[i][0].startswith("v_mfma")
    touched = [_regs(args) for _, args in code]
    found = []
    for i in range(len(code)):
        if mfma(i):
            mine, need = split(i), OPERANDS
            hit = lambda j: not mfma(j) and code[j][0].startswith("v_") and split(j)[0] & (mine[1] | mine[2] | mine[3])
        elif touched[i]:
            need = SUMS
            hit = lambda j: mfma(j) and split(j)[0] & touched[i]
        else:
            continue
        seen, todo = {}, [(j, 0) for j in before[i]]   # (what comes before, wait states between)
        while todo:
            j, d = todo.pop()
            if d >= need or seen.get(j, need) <= d:
                continue
            seen[j] = d
            if hit(j):
                found.append((d, code[j], code[i]))
                continue
            op, args = code[j]
            todo += [(k, d + (int(args) + 1 if op == "s_nop" else 1)) for k in before[j]]
    return found


def _assembly(name, tmp_path):
    out = tmp_path / (name + ".s")
    cmd = [_build._hipcc(), "-O3", "-std=c++17", f"--offload-arch={_build.ARCH}", "-fno-gpu-rdc", f"-I{_build.CSRC}", "-w", *_build._NO_PACKED_FP32,
           "--cuda-device-only", "-S", str(_build.CSRC / (name + ".hip")), "-o", str(out)]
    subprocess.run(cmd, check=True, stdout=subprocess.DEVNULL, stderr=subprocess.DEVNULL)
    return out.read_text()


@pytest.mark.parametrize("name", ["act_gemm", "grouped_rowgemm", "wgrad_gemm"])
def test_products_have_their_waits(name, tmp_path):
    kernels = {f: c for f, c in _functions(_assembly(name, tmp_path)).items() if any(op.startswith("v_mfma") for op, _ in c[0])}
    assert kernels
    for f, (code, labels) in kernels.items():
        assert not _close(code, labels)[:5], f


def test_stores_between_tiles_are_as_many_as_the_wait_says(tmp_path):
    """A tile's stores are in flight while the next tile's first step waits for the loads ahead of them by their count: vmcnt(8 + stores), in products whose workgroups
    have several tiles.  Fewer stores in its path would let it go on too early; registers in scratch memory would make that path another one."""
    asm = _assembly("act_gemm", tmp_path)
    assert set(re.findall(r"; ScratchSize: (\d+)", asm)) == {"0"}
    seen = {}
    for f, (code, labels) in _functions(asm).items():
        counts = {int(n) for op, args in code if op == "s_waitcnt" for n in re.findall(r"vmcnt\((\d+)\)", args)}
        several = counts & {8 + 16, 8 + 32}
        if several and any(op.startswith("v_mfma") for op, _ in code):
            edges = sorted({0, len(code), *labels.values(), *(i + 1 for i, (op, _) in enumerate(code) if op.startswith(("s_branch", "s_cbranch")))})
            # the path without checks: a straight line with more than one store
            lines = [[op for op, _ in code[a:b] if op.startswith(("global_", "flat_", "buffer_", "scratch_"))] for a, b in zip(edges, edges[1:])]
            seen[f] = (max(several), [ops for ops in lines if sum(op.startswith("global_store") for op in ops) > 1])
    assert len(seen) == 2
    for f, (wait, paths) in seen.items():
        assert [set(p) for p in paths] == [{"global_store_dwordx4"}] and len(paths[0]) == wait - 8, f


def test_what_is_too_near_is_found():
    near = "k:\n\tv_mfma_f32_16x16x32_bf16 a[0:3], v[0:3], v[4:7], a[0:3]\n\ts_nop {}\n\tv_accvgpr_read_b32 v9, a2\n"
    assert not _close(*_functions(near.format(7))["k"]) and _close(*_functions(near.format(6))["k"])
    moved = "k:\n\tv_accvgpr_write_b32 a3, v9\n{}\tv_mfma_f32_16x16x32_bf16 a[0:3], v[0:3], v[4:7], a[0:3]\n"
    assert _close(*_functions(moved.format("\ts_nop 0\n"))["k"]) and not _close(*_functions(moved.format("\ts_nop 1\n"))["k"])
    loop = "k:\n.L1:\n\tv_accvgpr_read_b32 v9, a2\n\tv_mfma_f32_16x16x32_bf16 a[0:3], v[0:3], v[4:7], a[0:3]\n\ts_cbranch_scc1 .L1\n\ts_endpgm\n"
    assert _close(*_functions(loop)["k"])
