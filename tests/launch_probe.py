"""What a GEMM call would launch, seen on the CPU: run as a program with the launch recorder preloaded, it reads a list of calls
as JSON and prints, for each, the statuses, the state and the launches.  launches() builds the recorder and runs it."""
import ctypes
import json
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))


def launches(tmp_path, calls):
    """calls: dicts of q, p, signed, M, N, K and optionally tile (a kernel name), layouts, group, zeros, act, row_sums, value_bits,
    workspace, dynamic (fp16 activations quantised in the kernel, last), tuning (lines of a tuning table), order (of the declarations), then
    (further ones: [what, value]); or pack: [rows, k, bits], a packing of int32 codes.  Returns a list of dicts: status, tile, strategy, grid, block, lds, launches."""
    so = str(tmp_path / "librecorder.so")
    if not os.path.exists(so):
        subprocess.check_call(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", os.path.join(HERE, "cpp", "launch_recorder.cpp"), "-o", so])
    env = dict(os.environ, LD_PRELOAD=so, RECORDER=so, CUDA_VISIBLE_DEVICES="", HIP_VISIBLE_DEVICES="")
    out = subprocess.run([sys.executable, os.path.abspath(__file__)], input=json.dumps(calls), capture_output=True, text=True, env=env, timeout=300)
    assert out.returncode == 0, out.stderr[-2000:]
    return json.loads(out.stdout.splitlines()[-1])


def main():
    sys.path.insert(0, HERE)
    from conftest import load_abq_gemm
    abq = load_abq_gemm()
    L = abq.lib()
    rec = ctypes.CDLL(os.environ["RECORDER"])
    rec.recorder_name.restype = ctypes.c_char_p

    def recorded():
        made = []
        for i in range(rec.recorder_count()):
            grid, block, lds = (ctypes.c_uint32 * 3)(), (ctypes.c_uint32 * 3)(), ctypes.c_uint64()
            rec.recorder_sizes(i, grid, block, ctypes.byref(lds))
            made.append({"kernel": rec.recorder_name(i).decode(), "grid": list(grid), "block": list(block), "lds": lds.value})
        return made

    def one(c):
        if "pack" in c:
            rec.recorder_clear()
            return {"status": L.abq_pack_i32(0x100000, 0x200000, *c["pack"], None), "launches": recorded()}
        L.abq_tuning_clear()
        for line in c.get("tuning", []):
            name, m, n, k, group, tops = line.split()
            cfg = abq.parse_kernel_name(name)[0]
            assert L.abq_tuning_add(ctypes.byref(cfg), int(m), int(n), int(k), int(group), float(tops)) == 0
        L.abq_tuning_enable_builtin(int(c.get("builtin", False)))
        st = abq.GemmState()
        s = ctypes.byref(st)
        tile = abq.parse_kernel_name(c["tile"])[0] if c.get("tile") else None
        group = c.get("group", 0)
        rc = [L.abq_gemm_init(ctypes.byref(tile) if tile else None, c["q"], c["p"], c["signed"], 0x100000, 0x200000, c["M"], c["N"], c["K"],
                              0x300000, 0x380000, 0, abq.OUT_F16_SCALED if group else c.get("out_kind", abq.OUT_I32), s)]
        steps = {"value_bits": lambda: L.abq_gemm_set_value_bits(s, *c["value_bits"]) if "value_bits" in c else 0,
                 "layouts": lambda: L.abq_gemm_set_operand_layout(s, *c.get("layouts", (abq.LAYOUT_TILED, abq.LAYOUT_TILED))),
                 "row_sums": lambda: L.abq_gemm_set_row_sums(s, *c["row_sums"]) if "row_sums" in c else 0,
                 "scales": lambda: L.abq_gemm_set_scales(s, 0x400000, 0x500000, group) if group or c.get("out_kind") == abq.OUT_F16_SCALED else 0,
                 "zeros": lambda: L.abq_gemm_set_zero_points(s, 0x600000, 0x700000, 0x800000, 0x900000) if c.get("zeros") else 0,
                 "act": lambda: L.abq_gemm_set_activation(s, c["act"]) if c.get("act") else 0,
                 "workspace": lambda: L.abq_gemm_set_workspace(s, 0xA00000, c["workspace"]) if c.get("workspace") else 0}
        for step in c.get("order", list(steps)):
            if rc[-1] == 0:
                rc.append(steps[step]())
        for what, value in c.get("then", []):
            c = dict(c, **{what: value})
            if rc[-1] == 0:
                rc.append(steps[what]())
        if c.get("dynamic") and rc[-1] == 0:
            rc.append(L.abq_gemm_set_dynamic_f16_activations(s, 0x100000, 1))
        rec.recorder_clear()
        if rc[-1] == 0:
            rc.append(L.abq_gemm_exec(s, None))
        made = recorded()
        d3 = lambda d: [d.x, d.y, d.z]  # noqa: E731
        return {"status": rc[-1], "tile": abq.format_kernel_name(st.cfg) if rc[0] == 0 else None, "strategy": abq.STRATEGY_NAMES[st.strategy],
                "grid": d3(st.grid_dim), "block": d3(st.block_dim), "lds": st.shared_mem_size, "launches": made}

    calls = json.load(sys.stdin)
    results = [one(c) for c in calls]
    text = "\n".join(l["kernel"] for r in results for l in r["launches"])
    names = iter(subprocess.run(["c++filt"], input=text, capture_output=True, text=True, check=True).stdout.splitlines()) if text else iter(())
    for r in results:
        for l in r["launches"]:
            l["kernel"] = next(names).split("(")[0].replace("void ", "").replace("abq::", "")
    print(json.dumps(results))


if __name__ == "__main__":
    main()
