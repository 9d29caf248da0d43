// sbz_rtc: compiles one HIP source with hiprtc in a process of its own (sbz_rtc.cpp starts it).
// Source on stdin, compile options as arguments; descriptor 3 receives the code object and 'K', or the
// compiler's log and 'E' (last, so that an output cut short has neither).  Not stdout: a library preloaded
// into the process may print there before main.
#include <hip/hiprtc.h>
#include <unistd.h>

#include <cstdlib>
#include <string>
#include <vector>

static bool write_all(int fd, const char* p, size_t n) {
    while (n > 0) {
        const ssize_t w = write(fd, p, n);
        if (w <= 0) return false;
        p += w;
        n -= (size_t)w;
    }
    return true;
}

int main(int argc, char** argv) {
    const int out = 3;
    (void)dup2(2, 1);   // what the compiler prints
    // a cached result may be one of a compile whose options did not take hold
    setenv("AMD_COMGR_CACHE", "0", 1);
    std::string src, log;
    std::vector<char> buf(1 << 16), code;
    for (ssize_t r; (r = read(0, buf.data(), buf.size())) > 0;) src.append(buf.data(), (size_t)r);
    hiprtcProgram prog;
    hiprtcResult r = hiprtcCreateProgram(&prog, src.c_str(), "sbz_model.hip", 0, nullptr, nullptr);
    if (r == HIPRTC_SUCCESS) {
        r = hiprtcCompileProgram(prog, argc - 1, const_cast<const char**>(argv + 1));
        size_t n = 0;
        if (r != HIPRTC_SUCCESS) {
            if (hiprtcGetProgramLogSize(prog, &n) == HIPRTC_SUCCESS && n > 0) {
                log.resize(n);
                (void)hiprtcGetProgramLog(prog, &log[0]);
            }
        } else if ((r = hiprtcGetCodeSize(prog, &n)) == HIPRTC_SUCCESS) {
            code.resize(n);
            r = hiprtcGetCode(prog, code.data());
        }
    }
    if (r != HIPRTC_SUCCESS && log.empty()) log = hiprtcGetErrorString(r);
    const bool ok = r == HIPRTC_SUCCESS;
    const std::string tag = std::string("sbz_rtc:") + (ok ? 'K' : 'E');
    const bool sent = write_all(out, ok ? code.data() : log.data(), ok ? code.size() : log.size()) &&
                      write_all(out, tag.data(), tag.size());
    return sent && ok ? 0 : 1;
}
