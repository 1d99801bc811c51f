"""The argument kinds the Python binding declares for the C entry points, against the header they are compiled from."""
import os
import re
import subprocess
import sys

from flash3dtransformer_amd.lib import pshattn


def test_declared_signatures_match_the_header():
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    text = re.sub(r"/\*.*?\*/", "", open(os.path.join(root, "include", "f3d_hip.h")).read(), flags=re.S)

    def kind(arg):
        if "*" in arg:
            return "p"
        return {"uint32_t": "u", "int": "i", "float": "f", "size_t": "Q"}[arg.replace("const ", "").split()[0]]
    found = {name: "".join(kind(a.strip()) for a in args.split(",") if a.strip() not in ("", "void"))
             for name, args in re.findall(r"\b(f3d_\w+)\s*\(([^()]*)\)\s*;", text)}
    assert len(found) > 40 and found == pshattn._SIGNATURES


def test_pooling_checks_its_tensors_once(monkeypatch):
    """the builder and the reduction of one pooling call read tensors that were checked together"""
    import torch
    seen = []
    monkeypatch.setattr(pshattn, "_lib", type("Lib", (), {"__getattr__": lambda self, name: lambda *a: 0})())
    monkeypatch.setattr(pshattn, "_stream", lambda dev: 0)
    monkeypatch.setattr(pshattn, "assert_same_device", lambda ts: 0)
    monkeypatch.setattr(pshattn, "assert_contiguous", lambda ts: seen.extend(id(t) for t in ts))
    u32, half, bf = [lambda *s, t=t: torch.zeros(*s, dtype=t) for t in (torch.uint32, torch.float16, torch.bfloat16)]
    off = torch.zeros(8, dtype=torch.uint16)
    box = half(3), half(3)
    pshattn.batch_subbuck_reduce(half(8, 3), bf(8, 16), u32(1), 8, 2, 0xFFFF, *box, u32(8), off, u32(1), half(4, 3), bf(4, 16), u32(4, 2), 1, 0,
                                 fill=True)
    assert len(seen) == len(set(seen)) == 11


def test_host_side_modules_import_on_a_torch_without_gpu_support():
    """such a torch has no raw stream call; sizes, planning and the layers' construction need none"""
    code = ("import torch; hasattr(torch._C, '_cuda_getCurrentRawStream') and delattr(torch._C, '_cuda_getCurrentRawStream')\n"
            "from flash3dtransformer_amd.psh import batching\n"
            "from flash3dtransformer_amd import layers\n"
            "print(batching.host_sizes(torch.tensor([3, 7])), layers.Linear(8, 4).weight.shape[0])")
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    got = subprocess.run([sys.executable, "-c", code], cwd=root, capture_output=True, text=True, timeout=300)
    assert got.returncode == 0 and got.stdout.split() == ["[3,", "4]", "4"], got.stderr[-2000:]
