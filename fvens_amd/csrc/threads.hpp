/* threads.hpp -- independent pieces of host work on threads.
 */
#ifndef FVX_THREADS_HPP
#define FVX_THREADS_HPP

#include <exception>
#include <thread>
#include <vector>

namespace fvx {

/// Runs f(0) .. f(nt - 1), on threads where they can be had; the first exception is rethrown when
/// all are done.
template <class F> void parallel(int nt, F&& f)
{
	std::vector<std::thread> th;
	std::vector<std::exception_ptr> err(nt);
	auto body = [&](int t) {
		try { f(t); } catch(...) { err[t] = std::current_exception(); }
	};
	th.reserve(nt);
	int t = 1;
	// no thread (std::system_error) or no memory for one: the rest runs here, those started are
	// joined below (destroying a running thread ends the process)
	try { for(; t < nt; t++) th.emplace_back(body, t); }
	catch(...) {}
	body(0);
	for(; t < nt; t++) body(t);
	for(std::thread& x : th) x.join();
	for(const std::exception_ptr& e : err) if(e) std::rethrow_exception(e);
}

}
#endif
