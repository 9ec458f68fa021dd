// RecordBlock (csrc/record_block.hpp) on a stand-in for the device: a table of
// one value a job.  Prints one line a scenario for tests/test_record_block_cpu.py.
#include <cstdio>
#include <memory>
#include <new>
#include <vector>

#include "../../mcrg_amd/csrc/record_block.hpp"

using mcrg::RecordBlock;

struct Device {
    std::vector<long long> value;
    RecordBlock ahead;
    int singles = 0, blocks = 0;
    bool no_memory = false, no_range = false, broken = false;

    explicit Device(int n) : value((size_t)n, 0) {}
    void advance(long long by)
    {
        for (long long &v : value) v += by;
    }
    int read(int job, long long &out)
    {
        return ahead.read<int>(
            job, reinterpret_cast<char *>(&out), sizeof(out),
            [&](int k) { return (size_t)(job + k) < value.size() ? sizeof(out) : 0u; },
            [&]() {
                ++singles;
                out = value[(size_t)job];
                return 0;
            },
            [&](int n, std::vector<size_t> &off, std::vector<char> &data) {
                if (no_memory) throw std::bad_alloc();
                if (broken) return 7;
                if (no_range) return 0;
                ++blocks;
                data.resize((size_t)n * sizeof(out));
                std::memcpy(data.data(), value.data() + job, data.size());
                for (int k = 0; k < n; ++k) off.push_back((size_t)k * sizeof(out));
                return 0;
            });
    }
    long long get(int job)
    {
        long long v = -1;
        const int e = read(job, v);
        return e == 0 ? v : -100 - e;
    }
};

int main()
{
    {
        Device d(3000);
        d.advance(5);
        bool same = true;
        for (int j = 0; j < 3000; ++j) same = same && d.get(j) == 5;
        std::printf("sequence same=%d singles=%d blocks=%d\n", same, d.singles, d.blocks);
    }
    {
        // another thread reads while a run is in progress, and again behind it
        Device d(100);
        std::printf("progress");
        {
            RecordBlock::Running run(d.ahead);
            d.advance(1);
            for (int j : {0, 1, 2, 3}) std::printf(" %lld", d.get(j));
            d.advance(1);
            for (int j : {1, 2, 3}) std::printf(" %lld", d.get(j));
            d.advance(1);
        }
        for (int j = 0; j < 6; ++j) std::printf(" %lld", d.get(j));
        std::printf("\n");
    }
    {
        // two runs that overlap: the first one's end is not the end
        Device d(100);
        auto a = std::make_unique<RecordBlock::Running>(d.ahead), b = std::make_unique<RecordBlock::Running>(d.ahead);
        a.reset();
        d.advance(1);
        for (int j : {0, 1, 2}) (void)d.get(j);
        d.advance(1);
        b.reset();
        std::printf("overlap");
        for (int j : {2, 3, 4}) std::printf(" %lld", d.get(j));
        std::printf("\n");
    }
    {
        // blocks read between runs are dropped by the next one
        Device d(100);
        for (int j = 0; j < 5; ++j) (void)d.get(j);
        {
            RecordBlock::Running run(d.ahead);
            d.advance(9);
        }
        std::printf("between");
        for (int j : {5, 6}) std::printf(" %lld", d.get(j));
        std::printf("\n");
    }
    {
        Device d(100);
        d.advance(4);
        std::printf("memory");
        for (int j = 0; j < 8; ++j) {
            d.no_memory = j < 3;
            d.no_range = j == 3 || j == 4;
            d.broken = j == 5;
            std::printf(" %lld", d.get(j));
        }
        std::printf("\n");
    }
    return 0;
}
