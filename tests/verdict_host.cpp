// The host side's verdicts over words that a test holds and fills in itself, for machines without a GPU: the operators' source as it
// is, and one function more.
#include "../gact-icml_amd/csrc/torch_ops.cpp"

namespace {
// verdict(int64[2] tensor) -> a verdict as batch_quantize makes it, of a plan launched on the first GPU's default stream
PyObject* verdict(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 1 || !THPVariable_Check(args[0])) Py_RETURN_NONE;
  Verdict* const v = new Verdict{THPVariable_Unpack(args[0]), c10::Device(c10::kCUDA, 0), nullptr};
  return PyCapsule_New(v, kVerdict, drop_verdict);
  END_HANDLE_TH_ERRORS
}
PyMethodDef host_methods[] = {FASTCALL(verdict), FASTCALL(verdict_wait), {nullptr, nullptr, 0, nullptr}};
PyModuleDef host_module = {PyModuleDef_HEAD_INIT, "verdict_host", "Verdicts without a GPU.", -1, host_methods};
}  // namespace

PyMODINIT_FUNC PyInit_verdict_host(void) { return PyModule_Create(&host_module); }
