"""The argument kinds the Python binding declares for the C entry points, against the header they are compiled from."""
import os
import re

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
