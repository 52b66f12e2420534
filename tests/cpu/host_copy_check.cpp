// host_copy_check.cpp -- copyOut (custen_amd/csrc/host_copy.h) over sizes around its
// splits, with all its threads and with memory for none to seven of them.
//
// prints "<copies> <wrong> <threads refused>"
#include <cstdio>
#include <cstdlib>
#include <new>
#include <vector>

#include "../../custen_amd/csrc/host_copy.h"

namespace {
bool counting = false;
int allowed = 0;  // allocations (one a thread) until memory is out
int refused = 0;
}  // namespace

void* operator new(std::size_t n)
{
    if (counting && allowed-- <= 0) {
        refused++;
        throw std::bad_alloc();
    }
    if (void* p = std::malloc(n)) return p;
    throw std::bad_alloc();
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, std::size_t) noexcept { std::free(p); }

int main()
{
    const size_t piece = 65536;  // 512 KB
    int copies = 0, wrong = 0;
    for (size_t count : std::vector<size_t>{0, 1, piece, 2 * piece - 1, 2 * piece, 2 * piece + 1,
                                            5 * piece + 7, 8 * piece, 40 * piece + 3}) {
        for (int threads = 0; threads <= 8; threads++) {
            std::vector<double> src(count + 1), dst(count + 1, -1.0);
            for (size_t i = 0; i <= count; i++) src[i] = (double)i;
            allowed = threads;
            counting = true;
            custen::copyOut(dst.data(), src.data(), count, 8);
            counting = false;
            copies++;
            bool same = dst[count] == -1.0;  // nothing past the end
            for (size_t i = 0; i < count; i++) same = same && dst[i] == src[i];
            wrong += !same;
        }
    }
    std::printf("%d %d %d\n", copies, wrong, refused);
    return 0;
}
