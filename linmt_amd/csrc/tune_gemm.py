"""Regenerates gemm_tuning.inc, the timing tables behind lh_gemm's choice of tile configuration.

Run on the target GPU from the repository root after any change to the GEMM kernel or its
configuration list, and rebuild:

    python linmt_amd/csrc/tune_gemm.py > new.inc && mv new.inc linmt_amd/csrc/gemm_tuning.inc
    python linmt_amd/csrc/tune_gemm.py NN:44 ragged-TN packed > new.inc     # these rows or blocks alone

With arguments (BLOCK or BLOCK:CONFIG) only those rows are timed and the others are taken from the
file as it is.  For every row it times a product whose tiles give each CU exactly one workgroup, and
one that gives each CU as many as fit at once, at two depths K; the table holds the fixed and per-k
cost of both, which is all the cost model in gemm.hip uses.  Blocks: the operand layouts NN, TN and
NT; "cell", the stacked gate product that ends in the LSTM cell; "ragged-NN", "ragged-TN" and
"ragged-NT", products of a few configurations where no row of an operand is 16-byte aligned; "narrow-NN" and
"narrow-TN", the tiles of 16 rows; "packed", the gate product with its cell on packed gate matrices.
"""
import os
import re
import sys
import textwrap

import torch

sys.path.insert(0, ".")
from linmt_amd import lib as lh  # noqa: E402

CUS = 256
KS = (512, 4096)
RAGGED_ROWS = (12, 15, 18)  # configurations whose form for ragged operands costs other than that for aligned ones
KS_RAGGED = (128, 2048)  # (no line holds from one slab of k to 4096: rows that share cache lines cost the more the deeper)
LAYOUTS = {"NN": (False, False), "TN": (True, False), "NT": (False, True)}
PLAIN = list(LAYOUTS)
BLOCKS = PLAIN + ["cell"] + ["ragged-" + lay for lay in PLAIN] + ["narrow-NN", "narrow-TN", "packed"]
FILE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "gemm_tuning.inc")


def timeit(fn, n=10, reps=7):
    """us of device time per call: the calls are replayed from a graph.  Issued one by one a short launch
    lasts as long as the host takes to issue it (8 us for the gate product with cell, where the GPU needs 4)."""
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        fn()
        stream.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            for _ in range(n):
                fn()
        graph.replay()
        best = 1e30
        for _ in range(reps):
            stream.synchronize()
            s, e = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            s.record()
            graph.replay()
            e.record()
            stream.synchronize()
            best = min(best, s.elapsed_time(e) / n * 1e3)
    return best


class Tuner:
    def __init__(self):
        self.L = lh.load()
        self.n_cfg = self.L.lh_gemm_set_config_override(-1)
        self.a = torch.randn(12288 * 4096 + 16384, device="cuda") * 0.05
        self.x = torch.randn(4096 * 4096 + 64, device="cuda") * 0.05
        self.c = torch.empty(12288 * 4096, device="cuda")
        self.bias, self.ones = torch.zeros(4 * 12288, device="cuda"), torch.ones(8192, dtype=torch.int32, device="cuda")

    def warm(self):
        """Brings the clocks up before the first measurement counts."""
        for _ in range(300):
            lh.gemm(4096, 4096, [(self.a, 4096, self.x, 2048, 2048)], self.c, 4096)
        torch.cuda.synchronize()

    def product(self, block, tiles_m, tiles_n, info, K):
        """The call to time, or None where the configuration does not run such a product."""
        a, x, c = self.a, self.x, self.c
        M, N = info["BM"] * tiles_m, info["BN"] * tiles_n
        if block in ("cell", "packed"):
            H = M // 4
            segs = [(a, 32 if block == "packed" else 4 * H, x, K, K)]
            call = lh.gate_gemm_lstm_cell_packed if block == "packed" else lh.gate_gemm_lstm_cell
            fn = lambda: call(H, N, segs, self.bias, c, self.ones, c, c[H * N:])  # noqa: E731
            try:
                fn()
            except lh.LinmtHipError:
                return None
            return fn
        tA, tX = LAYOUTS[block[-2:]]
        odd = 1 if block.startswith("ragged") else 0  # a leading dimension that keeps no row aligned
        # (transposed A: K is the odd extent, of both operands)
        segs = [(a, (K if tA else M) + odd, x, N if tX else K + (odd if tA else 0), K)]
        tile = "<%d, %d, %d, %d, %d, %d," % tuple(info[k] for k in ("BM", "BN", "WM", "WN", "WK", "BK"))
        name = lh.gemm_kernel_name(M, N, segs, tA, tX)
        if tile not in name or odd and name.count(",") != 8:  # (a ninth argument: the ragged form)
            return None
        return lambda: lh.gemm(M, N, segs, c, M, transA=tA, transX=tX)

    def row(self, block, cfg):
        """(resident workgroups, fixed us, us per k, the same with the CU full), None: not a row of this block."""
        layout = LAYOUTS[block[-2:]] if block[-2:] in LAYOUTS else (False, False)
        info = lh.gemm_config_info(cfg, *layout)
        # (the staged form that ragged operands take where aligned ones are streamed: not what the ring leaves room for)
        occ = max(1, info["occupancy"]) if not (block.startswith("ragged") and cfg == 15) else 1
        self.L.lh_gemm_set_config_override(cfg)
        fits = []
        for per_cu in (1, occ):
            tm, tn = 16 * per_cu, 16
            if info["BM"] == 16:  # the few columns that the narrow tiles are for
                tm, tn = (CUS * per_cu, 1) if block == "packed" else (CUS // 4 * per_cu, 4)
            while tm * info["BM"] > 12288:
                tm //= 2
                tn *= 2
            ts, depths = [], KS_RAGGED if block.startswith("ragged") else KS
            for K in depths:
                fn = self.product(block, tm, tn, info, K)
                if fn is None:
                    return None
                ts.append(timeit(fn))
            slope = (ts[1] - ts[0]) / (depths[1] - depths[0])
            fits += [max(0.0, ts[0] - slope * depths[0]), slope]
        return (occ, *fits)

    def configs(self, block):
        if block.startswith("ragged"):
            return RAGGED_ROWS
        if block.startswith("narrow"):
            return range(self.n_cfg, self.n_cfg + 2)
        return range(self.n_cfg + 2) if block == "packed" else range(self.n_cfg)


def rows_of_file():
    """{(block, configuration): row} of the present file."""
    rows, block = {}, None
    for line in open(FILE):
        block = (re.search(r"// block (\S+)", line) or [None, block])[1]
        m = re.search(r"\{(\d+), ([\d.]+)f, ([\d.]+)f, ([\d.]+)f, ([\d.]+)f\}.*// (\d+):", line)
        if m:
            rows[block, int(m[6])] = (int(m[1]), *(float(m[i]) for i in range(2, 6)))
    return rows


def main():
    asked = sys.argv[1:]
    for a in asked:
        if a.split(":")[0] not in BLOCKS:
            sys.exit(f"no block {a}: {', '.join(BLOCKS)}")
    t = Tuner()
    rows = rows_of_file() if asked else {}
    t.warm()
    try:
        for block in BLOCKS:
            for cfg in t.configs(block):
                if asked and block not in asked and f"{block}:{cfg}" not in asked:
                    continue
                rows.pop((block, cfg), None)
                r = t.row(block, cfg)
                if r:
                    rows[block, cfg] = r
                print(block, cfg, r, file=sys.stderr, flush=True)
    finally:
        t.L.lh_gemm_set_config_override(-1)

    def line(block, cfg, sparse):
        r = rows.get((block, cfg), (0, 0.0, 0.0, 0.0, 0.0))
        info = lh.gemm_config_info(cfg)
        text = "{%d, %.2ff, %.5ff, %.2ff, %.5ff}" % r
        text = "{%d, %s}" % (cfg, text) if sparse else text
        return f"        {text},  // {cfg}: {info['BM']}x{info['BN']} wk{info['WK']} bk{info['BK']}"

    print("// Written by tune_gemm.py on", torch.cuda.get_device_name(0))
    print("// {workgroups resident per CU, then (fixed us, us per k) with one workgroup per CU and")
    print("//  with the CU full}, timed by graph replays.")
    if asked:
        print("// The last run timed: " + "\n//   ".join(textwrap.wrap(" ".join(asked), 100)) + "\n// (the other rows are of earlier ones)")
    print(f"static_assert(kNumConfigs == {t.n_cfg}, \"gemm_tuning.inc is stale: rerun tune_gemm.py\");")
    print("const Tuning kTuning[4][kNumConfigs] = {")
    for block in PLAIN + ["cell"]:
        print(f"    {{  // block {block}" + (" (zeros: the configuration's LDS cannot hold a tile)" if block == "cell" else ""))
        for cfg in range(t.n_cfg):
            print(line(block, cfg, False))
        print("    },")
    print("};")
    for name, blocks in (("kRaggedTuning", ["ragged-" + lay for lay in PLAIN]),
                         ("kNarrowTuning", ["narrow-NN", "narrow-TN"]), ("kPackedTuning", ["packed"])):
        n = sum((blocks[0], cfg) in rows for cfg in range(t.n_cfg + 2))
        print("const TuningRow %s%s[%d] = {" % (name, "[%d]" % len(blocks) if len(blocks) > 1 else "", n))
        for block in blocks:
            if len(blocks) > 1:
                print(f"    {{  // block {block}")
            else:
                print(f"        // block {block}")
            for cfg in range(t.n_cfg + 2):
                if (block, cfg) in rows:
                    print(line(block, cfg, True))
            if len(blocks) > 1:
                print("    },")
        print("};")


if __name__ == "__main__":
    main()
