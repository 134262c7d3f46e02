// pgmg_readout.hip - level vectors from the device to host arrays.
#include "pgmg_internal.hpp"

#include <algorithm>
#include <condition_variable>
#include <cstring>
#include <thread>

namespace pgmg {

namespace {

const long long kChunk = 1 << 17;   // points a chunk
const int kCopiers = 8;             // threads that copy out of the chunks, at most

// What the copying threads share with the one that feeds them.
struct Feed {
	std::mutex mu;
	std::condition_variable filled, freed;
	int ready = 0;   // chunks filled by the device
	int taken = 0;   // chunks a thread has taken
	bool stop = false;
	int copied[HostReadout::kSlots];  // last chunk copied out of each slot
};

}  // namespace

HostReadout::~HostReadout() {
	if (own) hipHostFree(own);
	for (auto e : ev)
		if (e) hipEventDestroy(e);
}

// The device writes the points of a chunk straight into pinned memory, up to
// 8 chunks (1 MB each) ahead of the host threads that copy them on.  A host array is
// usually new, so its pages are mapped and cleared while it is filled: that,
// not the bus, bounds one thread (10 GB/s), and one chunk of each of up to 8
// threads is under way at a time.  Vectors of at most four chunks are copied
// by the caller: threads cost more than they save there.
// Into a new array: 257^3 (136 MB) 13.7 ms by hipMemcpy from a device copy, 3.8
// so; 161x130x147 (25 MB) 1.87 and 1.13; 33^3 57 and 39 us.  With 16 chunks 257^3
// takes 3.6 ms (then chunks of 0.5 MB: 4.4, of 2 MB: 3.8), but the buffer is pinned
// on a hierarchy's first read-out, which with 16 costs a 161x130x147 program
// 0.3 ms more.
hipError_t HostReadout::copy(hipStream_t s, const LevelView &L, const double *d, double *out) {
	std::lock_guard<std::mutex> one(mu);
	const long long N = (long long)L.m * L.n * L.o;
	const int nc = (int)((N + kChunk - 1) / kChunk);
	const int slots = std::min(nc, kSlots);
	const size_t need = sizeof(double) * (size_t)std::min(N, slots * kChunk);
	hipError_t e = hipSuccess;
	if (need > cap) {
		if (own) hipHostFree(own);
		own = buf = nullptr;
		cap = 0;
		e = hipHostMalloc((void **)&own, need, hipHostMallocDefault);
		if (e != hipSuccess) { own = nullptr; return e; }
		buf = own;
		cap = need;
	}
	for (int q = 0; q < slots; q++)
		if (!ev[q] && (e = hipEventCreateWithFlags(&ev[q], hipEventDisableTiming)) != hipSuccess) return e;

	const auto points = [&](int c) { return std::min(kChunk, N - c * kChunk); };
	const auto move_out = [&](int c) {
		memcpy(out + c * kChunk, buf + (c % slots) * kChunk, sizeof(double) * (size_t)points(c));
	};
	Feed f;
	for (int &c : f.copied) c = -1;
	std::thread copier[kCopiers];
	int threads = 0;
	if (nc > 4) {
		const int want = std::min({kCopiers, nc / 2, std::max(1, (int)std::thread::hardware_concurrency() - 1)});
		try {
			for (; threads < want; threads++)
				copier[threads] = std::thread([&] {
					std::unique_lock<std::mutex> lk(f.mu);
					for (;;) {
						f.filled.wait(lk, [&] { return f.stop || f.taken < f.ready; });
						if (f.taken >= f.ready) return;
						const int c = f.taken++;
						lk.unlock();
						move_out(c);
						lk.lock();
						f.copied[c % slots] = c;
						f.freed.notify_one();
					}
				});
		} catch (...) {  // no more threads to be had: go on with these
		}
	}
	int queued = 0;
	for (int c = 0; c < nc && e == hipSuccess; c++) {
		// a slot may be filled again once its last chunk is out; waits only
		// when nothing is under way on the device
		for (; queued < nc && e == hipSuccess; queued++) {
			if (queued >= slots) {
				std::unique_lock<std::mutex> lk(f.mu);
				const auto out_of = [&] { return f.copied[queued % slots] == queued - slots; };
				if (queued == c) f.freed.wait(lk, out_of);
				else if (!out_of()) break;
			}
			launch_unpack_vec(s, L, d, buf + (queued % slots) * kChunk, queued * kChunk, points(queued));
			e = hipEventRecord(ev[queued % slots], s);
		}
		if (e == hipSuccess) e = hipEventSynchronize(ev[c % slots]);
		if (e != hipSuccess) break;
		if (threads) {
			{
				std::lock_guard<std::mutex> lk(f.mu);
				f.ready = c + 1;
			}
			f.filled.notify_one();
		} else {
			move_out(c);
			f.copied[c % slots] = c;
		}
	}
	{
		std::lock_guard<std::mutex> lk(f.mu);
		f.stop = true;
	}
	f.filled.notify_all();
	for (int t = 0; t < threads; t++) copier[t].join();
	// what is still queued after an error writes to the buffer
	const hipError_t last = hipStreamSynchronize(s);
	return e != hipSuccess ? e : last;
}

}  // namespace pgmg
