// The exception of the host module, with the reference's text (csrc/kernels/exception.cuh:12-22).
#pragma once
#include <hip/hip_runtime_api.h>

#include <exception>
#include <string>
#include <utility>

namespace deep_ep {

class EPException : public std::exception {
    std::string message;

public:
    EPException(const char* name, const char* file, int line, const std::string& error) {
        message = std::string("Failed: ") + name + " error " + file + ":" + std::to_string(line) + " '" + error + "'";
    }
    explicit EPException(std::string text) : message(std::move(text)) {}
    const char* what() const noexcept override { return message.c_str(); }
};

inline void hip_check(hipError_t e, const char* file, int line) {
    if (e != hipSuccess) throw EPException("HIP", file, line, hipGetErrorString(e));
}

}  // namespace deep_ep
