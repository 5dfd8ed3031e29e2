// Stands in front of the HIP runtime in a process without a GPU and writes down what a library launches: kernels by name with
// their grid and block.  Nothing runs.  Loaded with global visibility before the library (tests/routes.py).
#include <cxxabi.h>

#include <cstdint>
#include <cstdlib>
#include <map>
#include <string>

namespace {

struct Dim3 {
    uint32_t x, y, z;
};
struct Launch {
    Dim3 grid, block;
    size_t shared;
    void* stream;
};

std::map<const void*, std::string>& kernels()
{
    static std::map<const void*, std::string> names;
    return names;
}
std::string log_text;
Launch pending;

}  // namespace

extern "C" {

void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*, int*)
{
    int status = 0;
    char* plain = abi::__cxa_demangle(name, nullptr, nullptr, &status);
    std::string s = plain != nullptr ? plain : name;
    std::free(plain);
    for (const char* part : {"(anonymous namespace)::", "ascq::", "void "}) {
        for (size_t at; (at = s.find(part)) != std::string::npos;) s.erase(at, std::char_traits<char>::length(part));
    }
    size_t end = 0;  // of the name: the first bracket outside the template arguments
    for (int depth = 0; end < s.size() && (depth > 0 || s[end] != '('); ++end) depth += s[end] == '<' ? 1 : s[end] == '>' ? -1 : 0;
    kernels()[host] = s.substr(0, end);
}
int __hipPushCallConfiguration(Dim3 grid, Dim3 block, size_t shared, void* stream)
{
    pending = Launch{grid, block, shared, stream};
    return 0;
}
int __hipPopCallConfiguration(Dim3* grid, Dim3* block, size_t* shared, void** stream)
{
    *grid = pending.grid;
    *block = pending.block;
    *shared = pending.shared;
    *stream = pending.stream;
    return 0;
}
int hipLaunchKernel(const void* kernel, Dim3 grid, Dim3 block, void**, size_t, void*)
{
    log_text += kernels()[kernel] + ";" + std::to_string(grid.x) + ";" + std::to_string(grid.y) + ";" + std::to_string(block.x) + "\n";
    return 0;
}
int hipGetLastError() { return 0; }

// the launches since the last call of this function, a line each: name;grid x;grid y;block
const char* launch_log_take()
{
    static std::string out;
    out.swap(log_text);
    log_text.clear();
    return out.c_str();
}

}  // extern "C"
