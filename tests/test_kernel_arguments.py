"""What one GEMM kernel alone is handed is no member of the arguments of all: a member more moves those behind it, and with
them the scalar loads of every other kernel."""

import re

from __graft_entry__ import PKG_DIR


def test_no_gemm_argument_is_the_k_split_kernels_alone():
    gemm = (PKG_DIR / "csrc" / "w8a8_gemm.h").read_text()
    body = re.search(r"struct GemmArgs \{\n(.*?)\n\};", gemm, re.S).group(1)
    decls = [line.split("//")[0] for line in body.split("\n")]
    members = [m for d in decls for m in re.findall(r"(\w+)\s*(?=[,;])", d)]
    assert len(members) >= 20
    start = gemm.index("void w8a8_gemm_ksplit_kernel(")
    end = gemm.index("\n}\n", start)
    others = gemm[:start] + gemm[end:] + "".join((PKG_DIR / "csrc" / f).read_text() for f in ("w8a8_gemm16.h", "w8a8_grouped.h"))

    def reads(text, member):
        return re.search(rf"\bg\.{member}\b", text)

    assert [m for m in members if reads(gemm[start:end], m) and not reads(others, m)] == []
