// Run-time compilation of emitted sources, each in a fresh child process (the program sbz_rtc beside
// this library).  The compiler's back end takes -sgpr-regalloc from its first compilation in a process
// and keeps it; options of others stay set as well.  In one process a source's code would depend on what
// was compiled before it, by this library or by any other user of hiprtc, and the kernels with one
// hierarchy per lane are wrong without that option.
#include <dlfcn.h>
#include <spawn.h>
#include <sys/mman.h>
#include <sys/wait.h>
#include <unistd.h>

#include <cerrno>
#include <cstring>
#include <string>
#include <vector>

#include "sbz_internal.h"

extern char** environ;

namespace {
struct Fd {   // an anonymous file
    int fd = memfd_create("sbz_rtc", MFD_CLOEXEC);
    ~Fd() {
        if (fd >= 0) close(fd);
    }
};
}  // namespace

int sbz_compile_hiprtc(const char* src, std::vector<char>& code) {
    // kernel_flags of symboltz/build.py
    const char* opts[] = {"--offload-arch=gfx950", "-O3", "-std=c++17", "-Xclang", "-target-feature", "-Xclang",
                          "-packed-fp32-ops", "-mllvm", "-disable-machine-licm", "-mllvm",
                          "-sgpr-regalloc=basic"};
    const int n_opts = (int)(sizeof(opts) / sizeof(opts[0])) - (std::strstr(src, "\n#define SBZ_GROUP_OK 1\n") ? 0 : 4);
    Dl_info lib;
    if (!dladdr(reinterpret_cast<const void*>(&sbz_compile_hiprtc), &lib) || !lib.dli_fname) {
        sbz_set_error("the library's own path is unknown: no way to its compiler program sbz_rtc");
        return SBZ_ERR_COMPILE;
    }
    std::string prog = lib.dli_fname;
    const size_t slash = prog.rfind('/');
    prog = (slash == std::string::npos ? std::string("./") : prog.substr(0, slash + 1)) + "sbz_rtc";
    Fd in, out;
    bool ok = in.fd >= 0 && out.fd >= 0;
    for (size_t n = std::strlen(src), at = 0; ok && at < n;) {
        const ssize_t w = pwrite(in.fd, src + at, n - at, (off_t)at);
        if (w > 0) at += (size_t)w;
        else ok = w < 0 && errno == EINTR;
    }
    if (!ok) {
        sbz_set_error("no memory for a source to compile: %s", std::strerror(errno));
        return SBZ_ERR_COMPILE;
    }
    std::vector<char*> argv{const_cast<char*>(prog.c_str())};
    for (int i = 0; i < n_opts; ++i) argv.push_back(const_cast<char*>(opts[i]));
    argv.push_back(nullptr);
    posix_spawn_file_actions_t fa;
    posix_spawn_file_actions_init(&fa);
    posix_spawn_file_actions_adddup2(&fa, in.fd, 0);
    posix_spawn_file_actions_adddup2(&fa, out.fd, 3);   // after stdin's: in.fd itself may be 3
    pid_t pid = 0;
    const int e = posix_spawn(&pid, prog.c_str(), &fa, nullptr, argv.data(), environ);
    posix_spawn_file_actions_destroy(&fa);
    if (e != 0) {
        sbz_set_error("cannot start the compiler program %s: %s", prog.c_str(), std::strerror(e));
        return SBZ_ERR_COMPILE;
    }
    int status = 0;   // not looked at: a caller may have SIGCHLD ignored, and the output says how it went
    while (waitpid(pid, &status, 0) < 0 && errno == EINTR) {}
    const off_t n = lseek(out.fd, 0, SEEK_END);
    code.resize(n > 0 ? (size_t)n : 0);
    for (size_t at = 0; at < code.size();) {
        const ssize_t r = pread(out.fd, code.data() + at, code.size() - at, (off_t)at);
        if (r > 0) at += (size_t)r;
        else if (r == 0 || errno != EINTR) code.clear();
    }
    std::string tag;
    const size_t nt = sizeof("sbz_rtc:K") - 1;
    if (code.size() >= nt) {
        tag.assign(code.end() - nt, code.end());
        code.resize(code.size() - nt);
    }
    if (tag != "sbz_rtc:K" || code.empty()) {
        const std::string log(code.begin(), code.end());
        sbz_set_error("hiprtc compile failed: %.900s", tag == "sbz_rtc:E" ? log.c_str() : "sbz_rtc ended early");
        code.clear();
        return SBZ_ERR_COMPILE;
    }
    return SBZ_OK;
}
