// Test driver for threads.hpp (built by tests/test_threads.py with g++):
//   threads_harness N K     parallel(N, ..) with the K-th allocation of the call refused (0: none);
//                           prints how often each piece ran, or "bad_alloc"
//   threads_harness N -P    piece P throws; prints the pieces that ran and the exception
#include "threads.hpp"
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <new>
#include <stdexcept>

static std::atomic<int> countdown{0};

void* operator new(size_t n)
{
	if(countdown > 0 && --countdown == 0) throw std::bad_alloc();
	void* p = std::malloc(n);
	if(!p) throw std::bad_alloc();
	return p;
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }

int main(int argc, char** argv)
{
	if(argc != 3) return 2;
	const int n = std::atoi(argv[1]), k = std::atoi(argv[2]);
	std::vector<std::atomic<int>> ran(n);
	const char* what = "";
	countdown = k > 0 ? k : 0;
	try {
		fvx::parallel(n, [&](int t) {
			ran[t]++;
			if(k < 0 && t == -k) throw std::runtime_error("piece");
		});
	}
	catch(const std::bad_alloc&) { what = "bad_alloc"; }
	catch(const std::runtime_error& e) { what = e.what(); }
	countdown = 0;
	for(int t = 0; t < n; t++) std::printf("%d ", (int)ran[t]);
	std::printf("%s\n", what);
	return 0;
}
