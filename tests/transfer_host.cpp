/* mpcd_transfer.h's copies on the CPU (tests/hip_double) */
#include "mpcd_transfer.h"

#include <cstdint>

namespace mpcdk {
void set_last_error(const std::string&) {}
}  // namespace mpcdk

/* One copy of n bytes (up 1: host to device, 0: back, -1: back with the wait
 * left to the caller).  type: the host array's
 * (hipMemoryType), strict: an unregistered pointer is an error to ask about.
 * Returns the number of wrong bytes once the stream has been waited for;
 * *copies: how many copies the runtime was given. */
extern "C" long long transfer_one(long long n, int up, int type, int strict, long long* copies) {
    std::vector<unsigned char> host((size_t)n + 64), dev((size_t)n + 64);
    std::vector<unsigned char>& src = up > 0 ? host : dev;
    std::vector<unsigned char>& dst = up > 0 ? dev : host;
    uint64_t r = 88172645463325252ull;
    for (long long i = 0; i < n; ++i) {
        r ^= r << 13;
        r ^= r >> 7;
        r ^= r << 17;
        src[(size_t)i] = (unsigned char)r;
        dst[(size_t)i] = (unsigned char)~r;
    }
    for (size_t i = (size_t)n; i < dst.size(); ++i) dst[i] = 0x5a;
    const std::vector<unsigned char> want(src.begin(), src.begin() + n);
    FakeRegistered& reg = fake_registered();
    reg = FakeRegistered{};
    reg.strict = strict != 0;
    if (type != hipMemoryTypeUnregistered) {
        reg.lo = (const char*)host.data();
        reg.hi = reg.lo + host.size();
        reg.type = (hipMemoryType)type;
    }
    FakeStream st;
    {
        mpcdk::HostCopy copy;
        if (up > 0) {
            copy.upload(dev.data(), host.data(), (size_t)n, &st);
            /* pageable memory may change on return */
            if (type == hipMemoryTypeUnregistered && st.queued > 1) std::fill(host.begin(), host.end(), 0);
        } else {
            const bool later = up < 0;
            const bool whole = later && copy.download_later(host.data(), dev.data(), (size_t)n, &st);
            if (!later) copy.download(host.data(), dev.data(), (size_t)n, &st);
            if ((st.done == st.queued) != (!later || whole)) return -1; /* complete on return, and only then */
        }
        (void)hipStreamSynchronize(&st);
    }
    *copies = st.queued;
    long long bad = 0;
    for (long long i = 0; i < n; ++i) bad += dst[(size_t)i] != want[(size_t)i];
    for (size_t i = (size_t)n; i < dst.size(); ++i) bad += dst[i] != 0x5a;
    return bad;
}
