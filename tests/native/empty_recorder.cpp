// empty_recorder.cpp — stands in for the torch operator behind at::empty (its mangled name, arguments unused), and
// counts its calls and those made while Python's global lock is held. Loaded with global symbols before the library's
// torch binding, so that the binding takes it; it allocates nothing: every call ends in a C++ exception.
#include <Python.h>

#include <stdexcept>

namespace {
int calls = 0, held = 0;
}

extern "C" {
void recorded_empty() __asm__(
    "_ZN2at4_ops19empty_memory_format4callEN3c108ArrayRefINS2_6SymIntEEESt8optionalINS2_10ScalarTypeEES6_INS2_"
    "6LayoutEES6_INS2_6DeviceEES6_IbES6_INS2_12MemoryFormatEE");
void recorded_empty() {
    ++calls;
    held += PyGILState_Check();
    throw std::runtime_error("recorded");
}
int empty_calls() { return calls; }
int empty_held() { return held; }
}
