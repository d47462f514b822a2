"""Regenerates gemm_tuning.inc, the timing table behind lh_gemm's choice of tile configuration.

Run on the target GPU from the repository root after any change to the GEMM kernel or its
configuration list:   python linmt_amd/csrc/tune_gemm.py > linmt_amd/csrc/gemm_tuning.inc
and rebuild.  For every configuration and operand layout it times a product whose tiles give each
CU exactly one workgroup, and one that gives each CU as many as fit at once, at two depths K; the
table holds the fixed and per-k cost of both, which is all the cost model in gemm.hip uses; a
fourth block does the same for the stacked gate product that ends in the LSTM cell, a fifth for that
product on packed gate matrices.
"""
import sys

import torch

sys.path.insert(0, ".")
from linmt_amd import lib as lh  # noqa: E402

CUS = 256
KS = (512, 4096)


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


def main():
    L = lh.load()
    n_cfg = L.lh_gemm_set_config_override(-1)
    a = torch.randn(12288 * 4096 + 64, device="cuda") * 0.05
    x = torch.randn(4096 * 4096 + 64, device="cuda") * 0.05
    c = torch.empty(12288 * 4096, device="cuda")
    # bring the clocks up before the first measurement counts
    warm = [(a, 4096, x, 2048, 2048)]
    for _ in range(300):
        lh.gemm(4096, 4096, warm, c, 4096)
    torch.cuda.synchronize()
    print("// Generated by tune_gemm.py on", torch.cuda.get_device_name(0))
    print("// {workgroups resident per CU, then (fixed us, us per k) with one workgroup per CU and")
    print("//  with the CU full}, by operand layout (NN, TN, NT) and configuration.")
    print(f"static_assert(kNumConfigs == {n_cfg}, \"gemm_tuning.inc is stale: rerun tune_gemm.py\");")
    print("const Tuning kTuning[5][kNumConfigs] = {")
    try:
        for lay, (tA, tX) in (("NN", (False, False)), ("TN", (True, False)), ("NT", (False, True))):
            print(f"    {{  // {lay}")
            for cfg in range(n_cfg):
                info = lh.gemm_config_info(cfg, tA, tX)
                occ = max(1, info["occupancy"])
                L.lh_gemm_set_config_override(cfg)
                fits = []
                for per_cu in (1, occ):
                    tm, tn = 16 * per_cu, 16
                    while tm * info["BM"] > 12288:
                        tm //= 2
                        tn *= 2
                    M, N = info["BM"] * tm, info["BN"] * tn
                    ts = []
                    for K in KS:
                        segs = [(a, K if tA else M, x, N if tX else K, K)]
                        ts.append(timeit(lambda: lh.gemm(M, N, segs, c, M, transA=tA, transX=tX)))
                    slope = (ts[1] - ts[0]) / (KS[1] - KS[0])
                    fits += [max(0.0, ts[0] - slope * KS[0]), slope]
                print(f"        {{{occ}, {fits[0]:.2f}f, {fits[1]:.5f}f, {fits[2]:.2f}f, {fits[3]:.5f}f}},"
                      f"  // {cfg}: {info['BM']}x{info['BN']} wk{info['WK']} bk{info['BK']}")
                sys.stdout.flush()
            print("    },")
        # the stacked gate product with the LSTM cell in its epilogue (a tile = BM/4 rows of each gate)
        bias, ones = torch.zeros(4 * 12288, device="cuda"), torch.ones(8192, dtype=torch.int32, device="cuda")
        for packed in (False, True):
            print("    {  // packed gate matrices with the cell epilogue (zeros: not a configuration of that kernel)"
                  if packed else
                  "    {  // NN with the cell epilogue (zeros: the configuration's LDS cannot hold a tile)")
            for cfg in range(n_cfg):
                info = lh.gemm_config_info(cfg, False, False)
                occ = max(1, info["occupancy"])
                L.lh_gemm_set_config_override(cfg)
                fits = []
                for per_cu in (1, occ):
                    tm, tn = 16 * per_cu, 16
                    while tm * info["BM"] > 12288:
                        tm //= 2
                        tn *= 2
                    H, B = info["BM"] // 4 * tm, info["BN"] * tn
                    ts = []
                    for K in KS:
                        segs = [(a, 32 if packed else 4 * H, x, K, K)]
                        if packed:
                            call = lh.gate_gemm_lstm_cell_packed
                            try:
                                call(H, B, segs, bias, c, ones, c, c[H * B:])
                            except lh.LinmtHipError:
                                break
                        else:
                            call = lh.gate_gemm_lstm_cell
                            if not lh.gate_gemm_lstm_cell_plan(H, B, segs)[0]:
                                break
                        ts.append(timeit(lambda: call(H, B, segs, bias, c, ones, c, c[H * B:])))
                    if len(ts) < 2:
                        break
                    slope = (ts[1] - ts[0]) / (KS[1] - KS[0])
                    fits += [max(0.0, ts[0] - slope * KS[0]), slope]
                if len(fits) < 4:
                    fits, occ = [0.0] * 4, 0
                print(f"        {{{occ}, {fits[0]:.2f}f, {fits[1]:.5f}f, {fits[2]:.2f}f, {fits[3]:.5f}f}},"
                      f"  // {cfg}: {info['BM']}x{info['BN']} wk{info['WK']} bk{info['BK']}")
                sys.stdout.flush()
            print("    },")
    finally:
        L.lh_gemm_set_config_override(-1)
    print("};")


if __name__ == "__main__":
    main()
