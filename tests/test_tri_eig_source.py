"""Reads csrc/tri_eig.hip. A kernel of the divide and conquer that has barriers must test the
status word through `failed`, which gives all threads of a workgroup one answer: another
workgroup of the same launch may clear the word meanwhile, and threads that left alone would
leave LDS entries unwritten that the others index memory with. Such a failure cannot be asked
for from outside (the solver fails on no finite matrix that is known), so the source is what is
checked."""
import re

from conftest import PKG


def kernels():
    text = re.sub(r"//[^\n]*", "", (PKG / "csrc" / "tri_eig.hip").read_text())
    for m in re.finditer(r"__global__[^;{]*?\b(tri_\w+)\s*\([^;{]*\)\s*\{", text):
        depth, i = 1, m.end()
        while depth:
            depth += {"{": 1, "}": -1}.get(text[i], 0)
            i += 1
        yield m.group(1), text[m.end():i]


def test_kernels_with_barriers_leave_together():
    seen = dict(kernels())
    with_status = [n for n, body in seen.items() if "w.info[1]" in body or "failed(w)" in body]
    assert {"tri_leaf_kernel", "tri_deflate_kernel", "tri_root_kernel", "tri_couple_kernel",
            "tri_vec_kernel"} <= set(with_status)
    for name in with_status:
        if "__syncthreads" in seen[name]:
            assert not re.search(r"w\.info\[1\]\s*==\s*0", seen[name]), name
