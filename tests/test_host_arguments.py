"""The launch calls' argument lists (spoc_amd._host) against what the caller's objects do meanwhile: the entry points are
replaced by functions of the test that look at what arrives, so no device is needed."""
import ctypes as C

import numpy as np
import pytest

NAMES = ("sarek_hip_execute_run_vectors", "sarek_hip_execute_run_source", "sarek_hip_execute_run_pipeline",
         "sarek_hip_last_run_path", "sarek_hip_fold_partials_f64")


@pytest.fixture
def entries(hip):
    """entries(name=function): those entry points call the function until the test ends."""
    def addresses(**replaced):
        return [C.cast(replaced.get(n, getattr(hip.lib, n)), C.c_void_p).value for n in NAMES]
    yield lambda **replaced: hip._host.bind(*addresses(**replaced))
    hip._host.bind(*addresses())


def stage_text(word, length=4000):
    """A text of its own (not interned, not shared)."""
    return "".join([word] * (length // len(word)))


def test_pipeline_keeps_the_stages_texts(hip, entries):
    """A stage given as a list may be changed by another thread while the library works on it: the text it was given is
    the one it reads."""
    from spoc_amd.sarek import Execute
    stage = [stage_text("first"), [Execute.Int(7)], (1, 1, 1), (1, 1, 1)]
    stages = [stage]
    want = stage[0].encode()
    seen, other = [], []

    @C.CFUNCTYPE(C.c_int, C.POINTER(hip.PipelineStage), C.c_int, C.POINTER(C.c_int))
    def run(given, n, launches):
        stage[0] = "gone"
        stages[0] = None
        other.extend(stage_text("other") for _ in range(64))     # takes the place of a text that was given back
        address = C.c_void_p.from_buffer(given.contents, hip.PipelineStage.ir_text.offset).value
        seen.append((C.string_at(address, len(want)), given.contents.n_args, given.contents.args[0].i32))
        return hip.OK
    entries(sarek_hip_execute_run_pipeline=run)
    Execute.run_pipeline(stages)
    assert seen == [(want, 1, 7)]


class Changes:
    """An integer that changes a list when it is asked for its value."""

    def __init__(self, value, change):
        self.value, self.change = value, change

    def __index__(self):
        self.change()
        return self.value


def test_arguments_are_those_the_list_held(hip, entries):
    """Whatever __index__ of an argument, or of a block's size, does to the list that is being read."""
    from spoc_amd.sarek import Execute
    args, block = [], []
    args += [("i32", Changes(1, args.clear)), ("i32", 2), ("i64", 3)]
    block += [Changes(8, block.clear), 4, 2]
    seen = []

    @C.CFUNCTYPE(C.c_int, C.c_char_p, C.POINTER(C.c_int), C.POINTER(C.c_int), C.c_int, C.POINTER(hip.VArg), C.c_int)
    def run(ir, block, grid, shared, given, n):
        seen.append((list(block[:3]), [given[0].i32, given[1].i32, given[2].i64], n))
        return hip.OK
    entries(sarek_hip_execute_run_vectors=run)
    Execute.run_vectors("(kernel)", args, block, (1, 1, 1))
    assert seen == [([8, 4, 2], [1, 2, 3], 3)]


@pytest.mark.parametrize("given,want", [(True, 1), (False, 0), (np.True_, 1), (np.False_, 0), (1.0, 1)])
def test_inject_lengths_is_any_truth_value_that_is_a_number(hip, entries, given, want):
    """What int() takes: a float too, and numpy's booleans without the warning that their __index__ gives."""
    from spoc_amd.sarek import Execute
    seen = []

    @C.CFUNCTYPE(C.c_int, C.c_char_p, C.c_int, C.c_char_p, C.c_void_p, C.c_void_p, C.c_int, C.c_int, C.c_void_p, C.c_int)
    def run(source, lang, name, block, grid, shared, inject, args, n):
        seen.append(inject)
        return hip.OK
    entries(sarek_hip_execute_run_source=run)
    Execute.run_source("text", "name", (1, 1, 1), (1, 1, 1), [], inject_lengths=given)
    assert seen == [want]
