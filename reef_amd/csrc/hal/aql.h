// Recorded launch sequences submitted as packets to a hardware queue of this library's own.
//
// A launch through the runtime costs the host 3-4 us and gives the kernel an argument block that was
// written a moment ago: the first read of it is a trip past every cache.  A model launches the same
// kernels with the same arguments on every pass, so a pass here is recorded once: the argument
// blocks are uploaded to device memory and stay there, and each launch is a 64-byte packet that is
// copied into the queue (16 ns) on every run.
#pragma once
#include <cstddef>
#include <cstdint>
#include <memory>
#include <string>

namespace reef {
namespace hal {

struct AqlCode;   // one code object, loaded on the device on first use
struct AqlPass;

// The code object of `path` (read now; modules with the same contents share one copy).  nullptr: unreadable.
std::shared_ptr<AqlCode> aql_code_from_file(const char* path);

struct AqlLaunch {
    AqlCode* code;
    const char* name;
    uint32_t grid[3], block[3], dyn_lds;   // grid in workgroups
    const void* kernarg;
    size_t kernarg_bytes;
};

// Whether packets can be submitted to `device` (set up on first call; REEF_HAL_AQL=0: no).
bool aql_available(int device);
// nullptr and *err on failure.  Every launch's block has `tail_bytes` of the caller's behind the arguments.
AqlPass* aql_pass_create(int device, const AqlLaunch* launches, size_t n, size_t tail_bytes, std::string* err);
bool aql_pass_block(AqlPass* p, size_t i, char** device, char** host, size_t* bytes, size_t* tail);
// Uploads the blocks.
bool aql_pass_commit(AqlPass* p, std::string* err);
// Runs the recorded launches one after the other and returns when the last has finished.
// false and *err when the queue reported an error.
bool aql_pass_run(AqlPass* p, std::string* err);
void aql_pass_destroy(AqlPass* p);

}  // namespace hal
}  // namespace reef
