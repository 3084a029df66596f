"""Runs calls of the C ABI against the stand-in for the HIP runtime and prints what they would have launched.

    python record.py launches.so libps_adam.so _lib.py < calls

``calls`` is a JSON list of ``{"entry", "rows", "numels", "gated", "grad_f32"}``: addresses of the four arrays of every chunk or
tensor (never followed), lengths, whether the step is decided on the device, and which tensors have binary32 gradients."""
import ctypes
import importlib.util
import json
import sys


class Dim3(ctypes.Structure):
    _fields_ = [("x", ctypes.c_uint32), ("y", ctypes.c_uint32), ("z", ctypes.c_uint32)]


class Launch(ctypes.Structure):
    _fields_ = [("name", ctypes.c_char_p), ("grid", Dim3), ("block", Dim3), ("lds", ctypes.c_size_t)]


STATE, WORK = 1 << 30, 1 << 31  # addresses that nothing follows either
SCRATCH = 1 << 29
RATES = (1e-3, 0.9, 0.999, 1e-8, 0.01)


def main():
    stub = ctypes.CDLL(sys.argv[1], ctypes.RTLD_GLOBAL)
    spec = importlib.util.spec_from_file_location("signatures", sys.argv[3])
    _lib = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(_lib)
    assert "torch" not in sys.modules  # it would bring the real runtime
    lib = ctypes.CDLL(sys.argv[2])
    assert ctypes.c_int.in_dll(stub, "n_registered").value > 0, "the library is bound to another runtime"
    for name, (res, args) in _lib.SIGNATURES.items():
        getattr(lib, name).restype, getattr(lib, name).argtypes = res, args
    assert lib.ps_adam_create(1, *RATES, 1, 0) == 0
    count, launches = ctypes.c_int.in_dll(stub, "n_launches"), (Launch * 4096).in_dll(stub, "launches")

    def call(entry, rows, numels, gated, grad_f32):
        n, table, sizes = len(rows), _lib.chunk_array(rows), (ctypes.c_size_t * len(rows))(*numels)
        state = STATE if gated else None
        if entry == "chunks":
            longest = max(numels)
            if gated:
                return lib.ps_adam_step_chunks_dynamic(1, 1e-3, 1e-8, 0.01, 1, table, n, longest, sizes, None, 1, state, None, 0, 1, None)
            return lib.ps_adam_step_chunks(1, 1, *RATES, 1, table, n, longest, sizes, None, 8.0, None)
        if entry == "scratch":  # a device-decided step over chunks, with scratch memory
            return lib.ps_adam_step_chunks_dynamic_scratch(1, 1e-3, 1e-8, 0.01, 1, table, n, max(numels), sizes, None, 1, state, None, 0, 1, SCRATCH, 448, None)
        if entry == "tensors":
            return lib.ps_adam_step_tensors(1, 1, *RATES, 1, table, sizes, n, None, 8.0, state, None)
        if entry == "each":
            each = (_lib.ps_tensor_call * n)(*[(*RATES, 0 if gated else 1, -1, int(f)) for f in grad_f32])
            return lib.ps_adam_step_tensors_each(1, 1, table, sizes, each, n, 8.0, state, WORK, 64 * n, None)
        if entry == "dynamic":  # a whole device-decided step over tensors, which are probed as chunks; one set of numbers
            each = (_lib.ps_tensor_call * n)(*[(*RATES, 0, -1, 0)] * n)
            rc = lib.ps_adam_step_tensors_dynamic(1, 1, table, n, max(numels), sizes, table, sizes, each, n, state, None, 0, n, WORK, 64 * n, SCRATCH, 448, None)
            opened = count.value > 0 and b"open_planned" in launches[0].name
            assert lib.ps_tensors_at_once(table, n, max(numels), sizes, table, sizes, n) == opened
            return rc
        if entry == "operator":
            p, m, v, h = rows[0]
            return lib.ps_adam_update(1, 1, *RATES, 1, p, h, 1, m, v, numels[0], 8.0, None, None)
        raise KeyError(entry)

    out = []
    for one in json.load(sys.stdin):
        count.value = 0
        rc = call(**one)
        assert rc == 0, (rc, lib.ps_last_error())
        out.append([(q.name.decode(), [q.grid.x, q.grid.y], q.lds) for q in launches[: count.value]])
    json.dump(out, sys.stdout)


main()
