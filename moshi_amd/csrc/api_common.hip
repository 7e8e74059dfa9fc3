// Version / error plumbing of the C ABI (include/moshi_mi.h).
#include "mmi_common.h"
#include <mutex>

static thread_local std::string g_last_error;

void mmi_set_error(const std::string& msg) { g_last_error = msg; }
int mmi_fail(int code, const std::string& msg) {
    if (code == MMI_ERR_HIP) (void)hipGetLastError();       // reported here: the next launch check, ours or the caller's, must not find it again
    g_last_error = msg;
    return code;
}

extern "C" int mmi_version(void) { return MMI_ABI_VERSION; }
extern "C" const char* mmi_last_error(void) { return g_last_error.c_str(); }

// ---- device memory (mmi_common.h) --------------------------------------------------------------------------------------
static std::mutex g_unfreed_mu;
static std::vector<void*>& unfreed() {                     // (never destroyed: handles may outlive this file's statics)
    static std::vector<void*>* list = new std::vector<void*>;
    return *list;
}
static void free_unfreed() {
    std::lock_guard<std::mutex> g(g_unfreed_mu);
    std::vector<void*>& list = unfreed();
    while (!list.empty()) {
        if (hipFree(list.back()) != hipSuccess) {
            (void)hipGetLastError();
            return;
        }
        list.pop_back();
    }
}
static bool (*g_let_go)(int device) = nullptr;
void mmi_set_let_go(bool (*let_go)(int device)) { g_let_go = let_go; }
hipError_t mmi_malloc(void** p, size_t bytes) {
    free_unfreed();
    const hipError_t e = hipMalloc(p, bytes);
    int device = -1;
    if (e != hipErrorOutOfMemory || !g_let_go || hipGetDevice(&device) != hipSuccess || !g_let_go(device)) return e;
    (void)hipGetLastError();
    return hipMalloc(p, bytes);
}
void mmi_free(void* p) {
    free_unfreed();
    if (!p || hipFree(p) == hipSuccess) return;
    (void)hipGetLastError();
    std::lock_guard<std::mutex> g(g_unfreed_mu);
    unfreed().push_back(p);
}

// ---- launch-list recorder (mmi_graph.h) ------------------------------------------------------------------------------
static thread_local std::vector<std::string>* g_rec_log = nullptr;
static thread_local const char* g_rec_site = "-";
static thread_local long g_rec_bytes = 0;

void mmi_record_begin(std::vector<std::string>* log) { g_rec_log = log; g_rec_site = "-"; }
void mmi_record_site(const char* site) { g_rec_site = site; }
void mmi_record_bytes(long bytes) { g_rec_bytes = bytes; }
void mmi_record_end() { g_rec_log = nullptr; }
void mmi_note_launch(const char* kernel) {
    if (!g_rec_log) return;
    std::string k(kernel);
    while (!k.empty() && (k.front() == '(' || k.front() == ' ')) k.erase(k.begin());      // "(k_gemm_xp<...>)" -> "k_gemm_xp"
    const size_t cut = k.find_first_of("<)");
    if (cut != std::string::npos) k.resize(cut);
    std::string line = std::string(g_rec_site) + "\t" + k;
    if (g_rec_bytes > 0) line += "\t" + std::to_string(g_rec_bytes);
    g_rec_bytes = 0;
    g_rec_log->push_back(line);
}

// copy a launch log ("site\tkernel\n" per launch) into a caller buffer; returns the bytes needed (incl. the final NUL)
int64_t mmi_copy_launch_log(const std::vector<std::string>& log, char* buf, int64_t cap) {
    std::string all;
    for (const auto& l : log) { all += l; all += '\n'; }
    const int64_t need = (int64_t)all.size() + 1;
    if (buf && cap > 0) {
        const int64_t n = need <= cap ? need - 1 : cap - 1;
        memcpy(buf, all.data(), (size_t)n);
        buf[n] = 0;
    }
    return need;
}
