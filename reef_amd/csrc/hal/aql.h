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
struct AqlKernel; // one of its kernels

// The code object of `path` (read now; modules with the same contents share one copy).  nullptr: unreadable.
std::shared_ptr<AqlCode> aql_code_from_file(const char* path);

// A kernel of `code` (loaded on `device` if it is not yet), valid as long as the code is.  nullptr and *err: not found.
const AqlKernel* aql_kernel(AqlCode* code, int device, const char* name, std::string* err);
// One launch of `groups` workgroups of `threads`, waited for: it sees what finished kernels have written --
// and, `fresh`, what anybody else has (the caller's copies are other agents' stores to the device, which an acquire at
// agent scope promises nothing of) -- and its results are visible everywhere when this returns.  Calls of several
// threads run beside each other.
bool aql_call(int device, const AqlKernel* kernel, uint32_t groups, uint32_t threads, const void* kernarg, size_t kernarg_bytes,
              bool fresh, std::string* err);
// Makes what one call in flight needs, so that a first call allocates nothing (one beside another does).
bool aql_call_prepare(int device, std::string* err);

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
// Adds a last launch that copies device ranges to host memory of the pass's: host[i] for range i.  The first call
// allocates that memory, `reserve` bytes or more; a later one mirrors other ranges that fit into it.
bool aql_pass_mirror(AqlPass* p, int device, const void* const* src, const size_t* bytes, size_t n, size_t reserve, const char** host,
                     std::string* err);
// Runs the recorded launches one after the other and returns when the last has finished.
// fresh: the first launch drops what the caches hold of memory that others than finished kernels have
// written -- the host, the runtime's copies, aql_pass_commit (3 us: code and weights are fetched anew as well).
// false and *err when the queue reported an error.
bool aql_pass_run(AqlPass* p, bool fresh, std::string* err);
void aql_pass_destroy(AqlPass* p);

// Stores into device memory through the PCIe window, 45 GB/s; all of it has arrived when this returns.
// Caches may still hold the old bytes.  false: the device says nothing of how to flush the window.
bool aql_host_write(int device, void* dst, const void* src, size_t bytes);
// Copies device ranges to pinned host memory, one behind the other at multiples of 256 bytes, and waits for it: what
// kernels have written, and what others have in front of the last aql_fence.
bool aql_fetch(int device, const void* const* src, const size_t* bytes, size_t n, char* host, std::string* err);
// Drops what the caches hold of bytes that the host or the runtime's copies have replaced.
bool aql_fence(int device, std::string* err);

}  // namespace hal
}  // namespace reef
