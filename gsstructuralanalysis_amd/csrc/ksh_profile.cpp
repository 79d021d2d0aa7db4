// ksh_profile.cpp -- optional per-kernel timing with HIP events recorded on the launching stream.
//
// When enabled, each launcher brackets its kernel with a pair of events from a recycled pool;
// ksh_profile_query() waits for the pending pairs and accumulates hipEventElapsedTime per kernel.  The
// pairs of a stream are read before it is destroyed: an event recorded on a destroyed stream counts for one
// of whatever stream lives at its address later, and asking for it fails, and ends a capture there.
#include <hip/hip_runtime.h>

#include <map>
#include <mutex>
#include <string>
#include <vector>

#include "ksh_internal.hpp"
#include "ksh_profile.hpp"

namespace ksh {

namespace {

struct Pending {
    hipEvent_t start, stop;
    hipStream_t stream;
};
struct Entry {
    std::vector<Pending> pending;
    double total_ms = 0.0;
    long long count = 0;
    double work = 0.0;
};

std::mutex g_mu;
bool g_on = false;
std::map<std::string, Entry> g_entries;
std::vector<hipEvent_t> g_pool;

hipEvent_t take_event()
{
    if (!g_pool.empty()) {
        hipEvent_t e = g_pool.back();
        g_pool.pop_back();
        return e;
    }
    hipEvent_t e = nullptr;
    (void)hipEventCreate(&e);
    return e;
}

// reads the pending pairs of one stream, or all of them
void drain(Entry &en, const hipStream_t *stream = nullptr)
{
    std::vector<Pending> rest;
    for (auto &pr : en.pending) {
        if (stream && pr.stream != *stream) {
            rest.push_back(pr);
            continue;
        }
        (void)hipEventSynchronize(pr.stop);
        float ms = 0.f;
        if (hipEventElapsedTime(&ms, pr.start, pr.stop) == hipSuccess) {
            en.total_ms += ms;
            en.count += 1;
        }
        g_pool.push_back(pr.start);
        g_pool.push_back(pr.stop);
    }
    en.pending.swap(rest);
}

}  // namespace

bool profiling() { return g_on; }

void prof_count(const char *name, long long n)
{
    if (!g_on || n == 0) return;
    std::lock_guard<std::mutex> lk(g_mu);
    g_entries[name].count += n;
}

void destroy_stream(hipStream_t s)
{
    if (!s) return;
    {
        std::lock_guard<std::mutex> lk(g_mu);
        for (auto &kv : g_entries) drain(kv.second, &s);
    }
    (void)hipStreamDestroy(s);
}

ProfScope::ProfScope(const char *name, hipStream_t s) : m_name(name), m_stream(s)
{
    if (!g_on) return;
    std::lock_guard<std::mutex> lk(g_mu);
    m_start = take_event();
    m_stop = take_event();
    (void)hipEventRecord(m_start, s);
    m_active = true;
}

ProfScope::~ProfScope()
{
    if (!m_active) return;
    std::lock_guard<std::mutex> lk(g_mu);
    (void)hipEventRecord(m_stop, m_stream);
    Entry &en = g_entries[m_name];
    en.pending.push_back({m_start, m_stop, m_stream});
    en.work += m_work;
}

}  // namespace ksh

extern "C" {

int ksh_profile_enable(int on)
{
    std::lock_guard<std::mutex> lk(ksh::g_mu);
    ksh::g_on = on != 0;
    return KSH_SUCCESS;
}

int ksh_profile_reset(void)
{
    std::lock_guard<std::mutex> lk(ksh::g_mu);
    for (auto &kv : ksh::g_entries) ksh::drain(kv.second);
    ksh::g_entries.clear();
    return KSH_SUCCESS;
}

int ksh_profile_query(const char *kernel, int64_t *launches, double *total_ms)
{
    if (!kernel) return ksh::fail(KSH_OTHER_ERROR, "null argument");
    std::lock_guard<std::mutex> lk(ksh::g_mu);
    auto it = ksh::g_entries.find(kernel);
    if (it == ksh::g_entries.end()) {
        if (launches) *launches = 0;
        if (total_ms) *total_ms = 0.0;
        return KSH_SUCCESS;
    }
    ksh::drain(it->second);
    if (launches) *launches = it->second.count;
    if (total_ms) *total_ms = it->second.total_ms;
    return KSH_SUCCESS;
}

int ksh_profile_query_work(const char *kernel, double *work)
{
    if (!kernel || !work) return ksh::fail(KSH_OTHER_ERROR, "null argument");
    std::lock_guard<std::mutex> lk(ksh::g_mu);
    auto it = ksh::g_entries.find(kernel);
    *work = it == ksh::g_entries.end() ? 0.0 : it->second.work;
    return KSH_SUCCESS;
}

}  // extern "C"
