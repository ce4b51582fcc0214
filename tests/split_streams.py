"""Run as a script by tests/test_gpu_split.py: wide rows of small batches on a caller's streams (torch's) and
in a captured graph. Alternating streams without waits in between, and replays of a graph with other calls
of the same context between them, must give the ids of the same calls made one at a time."""
import os
import sys

import torch  # must precede voxwerk_amd

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, REPO)

import numpy as np  # noqa: E402

from voxwerk_amd._lib import PARAMS_DTYPE  # noqa: E402
from voxwerk_amd.sampler import Context  # noqa: E402

ROWS, VOCAB = 12, 60000


def main() -> int:
    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(5)
    p = np.zeros(ROWS, dtype=PARAMS_DTYPE)
    p["do_sample"], p["top_p"], p["temperature"], p["rep_penalty"] = 1, np.float32(0.9), 1.0, 1.0
    p["top_k"] = [0, 50] * (ROWS // 2)
    p["keep_id"], p["ban_id"] = -1, -1
    params = torch.from_numpy(p.view(np.uint8).copy()).to(dev)
    calls = [(torch.randn((ROWS, VOCAB), generator=g, device=dev) * 2, torch.rand(ROWS, generator=g, device=dev, dtype=torch.float64))
             for _ in range(12)]

    def sample(ctx, i, out):
        x, u = calls[i]
        ctx.sample_device(ROWS, VOCAB, x, VOCAB, params, 1, u, out)

    with Context(0) as ctx:
        want = []
        for i in range(len(calls)):
            out = torch.full((ROWS,), -99, dtype=torch.int32, device=dev)
            sample(ctx, i, out)
            ctx.synchronize()
            want.append(out.cpu())
        torch.cuda.synchronize()
        streams = [torch.cuda.Stream() for _ in range(6)]  # more than the context holds workspaces for
        for turn in range(3):
            outs = [torch.full((ROWS,), -99, dtype=torch.int32, device=dev) for _ in calls]
            torch.cuda.synchronize()
            for i in range(len(calls)):
                ctx.set_stream(streams[(i + turn) % len(streams)].cuda_stream)
                sample(ctx, i, outs[i])
            ctx.set_stream(None)
            torch.cuda.synchronize()
            bad = [i for i in range(len(calls)) if not torch.equal(outs[i].cpu(), want[i])]
            print(f"streams turn {turn}: {len(bad)} of {len(calls)} differ", flush=True)
            if bad:
                return 1
        out = torch.full((ROWS,), -99, dtype=torch.int32, device=dev)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            ctx.set_stream(torch.cuda.current_stream().cuda_stream)
            sample(ctx, 3, out)
            ctx.set_stream(None)
        for rep in range(4):
            out.fill_(-99)
            other = torch.full((ROWS,), -99, dtype=torch.int32, device=dev)
            torch.cuda.synchronize()
            graph.replay()
            sample(ctx, rep, other)
            torch.cuda.synchronize()
            print(f"replay {rep}", flush=True)
            if not torch.equal(out.cpu(), want[3]) or not torch.equal(other.cpu(), want[rep]):
                return 1
    return 0


if __name__ == "__main__":
    sys.exit(main())
