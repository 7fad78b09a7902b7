"""A batch's kernels read a scene's Dev from memory and declare each of its pointers as one to global
memory by name: a pointer left off the list would be read, and used, as a flat one."""
import os
import re

from natray_amd.build import CSRC


def test_every_pointer_of_dev_is_listed_once():
    text = open(os.path.join(CSRC, "natray_dev.h")).read()
    body = text[text.index("struct Dev {"):]
    body = re.sub(r"//[^\n]*", "", body[:body.index("\n};")])
    declared = [m for line in body.split(";") for m in re.findall(r"\*\s*(\w+)", line)]
    macro = text[text.index("#define NATRAY_DEV_POINTERS(X)"):]
    listed = re.findall(r"X\((\w+)\)", macro[macro.index("\n"):macro.index("\n\n")])
    assert len(declared) > 40
    assert sorted(listed) == sorted(declared)


def test_a_dev_is_filled_by_bytes():
    """No store into a Dev through a pointer to another type, which its later reads need not see."""
    text = open(os.path.join(CSRC, "natray_kernels.hip")).read()
    body = text[text.index("__device__ __forceinline__ Dev load_dev("):]
    body = body[:body.index("\n}")]
    assert not re.search(r"reinterpret_cast<(?!\s*(?:const\s+)?char\s*\*)[^>]*>\(&d\)", body)
