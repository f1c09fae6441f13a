// Stand-ins of the prover core for the proof service's CPU tests: service.hip is
// compiled as host code and linked with these instead of the runtime.  A core is a
// token, a program the number of milliseconds that a round of it takes, and every
// job ends with its first round.
#include <sys/resource.h>
#include <chrono>
#include <cstdint>
#include <cstdlib>
#include <string>
#include <thread>
#include <vector>
#include <hip/hip_runtime.h>
#include "sqd.h"

struct sqd_program {
    unsigned ms;
};
struct sqd_core {
    const sqd_program* prog;
    uint64_t rows;
};

namespace sqd {
void set_last_error(const std::string&) {}
}
extern "C" {
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDeviceProperties(hipDeviceProp_t*, int) { return hipErrorNoDevice; }
const char* sqd_last_error(void) { return ""; }
void sqd_settings_default(sqd_settings* s) { *s = sqd_settings{}; }
int sqd_program_nargs(const sqd_program*) { return 1; }
int sqd_core_create(int, const sqd_program* p, const sqd_settings*, sqd_core** out) {
    *out = new sqd_core{p, 0};
    return SQD_OK;
}
void sqd_core_destroy(sqd_core* c) { delete c; }
int sqd_core_memory(const sqd_core*, uint64_t* bytes) { *bytes = 0; return SQD_OK; }
int sqd_core_shape(const sqd_core*, uint32_t*, uint32_t*) { return SQD_ERR_INTERNAL; }
int sqd_batch_admit(sqd_core* c, uint32_t row, uint32_t, uint32_t) {
    c->rows |= 1ull << row;
    return SQD_OK;
}
int sqd_batch_step(sqd_core* c, sqd_job_counts*, uint64_t* finished, uint32_t* active) {
    std::this_thread::sleep_for(std::chrono::milliseconds(c->prog->ms));
    *finished = c->rows;
    *active = 0;
    c->rows = 0;
    return SQD_OK;
}
int sqd_batch_frontier(sqd_core*, uint64_t* counts, size_t n) {
    for(size_t i = 0; i < n; ++i) counts[i] = 0;
    return SQD_OK;
}
int sqd_prove_batch(sqd_core*, size_t, const uint32_t*, const uint32_t*, sqd_job_counts*, double*) { return SQD_ERR_INTERNAL; }
int sqd_prove_range(sqd_core*, uint32_t, uint32_t, sqd_counts*, double*, double*, size_t, size_t*, double*) {
    return SQD_ERR_INTERNAL;
}

// Runs one job of each of `programs` programs, the first of `ms` milliseconds and the
// others of 1, on a service with a worker per program and memory for one core.
// Returns how often a thread of the process gave up its processor meanwhile, or -1.
long service_waits(unsigned programs, unsigned ms) {
    sqd_service_options opt;
    sqd_service_options_default(&opt);
    opt.workers = programs;
    opt.batch_jobs = 1;
    opt.core_bytes_estimate = 1000;
    opt.memory_budget = 1000;
    sqd_service* s = nullptr;
    if(sqd_service_create(&opt, &s) != SQD_OK) return -1;
    std::vector<sqd_program> progs(programs, sqd_program{1});
    progs[0].ms = ms;
    std::vector<uint64_t> jobs(programs);
    rusage before{}, after{};
    getrusage(RUSAGE_SELF, &before);
    bool ok = true;
    for(unsigned i = 0; i < programs; ++i) {
        ok = ok && sqd_service_submit(s, &progs[i], 0, 1, &jobs[i]) == SQD_OK;
        if(i == 0) std::this_thread::sleep_for(std::chrono::milliseconds(5));   // it takes the only core
    }
    for(uint64_t j : jobs) ok = sqd_service_wait(s, j, nullptr) == SQD_OK && ok;
    getrusage(RUSAGE_SELF, &after);
    sqd_service_destroy(s);
    return ok ? after.ru_nvcsw - before.ru_nvcsw : -1;
}
}
