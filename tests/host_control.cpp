// What two kernels leave behind for the tests on host_runtime.c: k_control, the control block of an
// increment whose iterations stop after `stop` of them, and k_reduce at an increment's end, sums of zero.
#include "../srx_amd/csrc/srx_dev.hpp"

extern "C" void host_control(void *block, int stop) {
    srx::IterCtl &c = *static_cast<srx::IterCtl *>(block);
    if (c.done) return;
    c.iter += 1;
    c.s_vm = 1.0;
    c.done = c.iter >= stop;
    if (c.done && c.done_host) *c.done_host = 1;
}

extern "C" void host_reduce(int nvals, double *out) {
    for (int k = 0; nvals == srx::END_NPART && k < nvals; ++k) out[k] = 0.0;
}
