// Which threads are launching calls that had been put aside, for a thread that is about to give device memory back and has to come
// behind those launches.
#pragma once

#include <algorithm>
#include <atomic>
#include <memory>
#include <mutex>
#include <thread>
#include <utility>
#include <vector>

namespace nh {

// A thread writes into a word of its own when it goes in and out; who waits looks at all of them once and then waits for those that were inside,
// not for any that go in meanwhile: with a lock that those inside share, a thread that gave memory back beside seven that launched all the time
// waited 6 ms on average and up to 50, and whoever took another lock inside depended on that lock letting new ones in beside one who waits.
class CLaunchGate {
	typedef std::atomic<unsigned long long> CEntries; // odd: inside

public:
	// a thread's place, made and destroyed by that thread
	class CThread {
	public:
		explicit CThread( CLaunchGate& _gate ) : gate( _gate ), entries( std::make_shared<CEntries>( 0 ) )
		{
			std::lock_guard<std::mutex> guard( gate.lock );
			gate.threads.push_back( entries );
		}
		~CThread()
		{
			std::lock_guard<std::mutex> guard( gate.lock );
			gate.threads.erase( std::find( gate.threads.begin(), gate.threads.end(), entries ) );
		}
		CThread( const CThread& ) = delete;
		CThread& operator=( const CThread& ) = delete;

		// ( in turn )
		void Enter() { entries->fetch_add( 1 ); }
		void Leave() { entries->fetch_add( 1 ); }

	private:
		CLaunchGate& gate;
		const std::shared_ptr<CEntries> entries;
	};

	// until every thread that is inside now has left; by a thread that is not
	void WaitForThoseInside()
	{
		std::vector<std::pair<std::shared_ptr<CEntries>, unsigned long long>> inside;
		{
			std::lock_guard<std::mutex> guard( lock );
			for( const auto& thread : threads ) {
				const unsigned long long seen = thread->load();
				if( seen % 2 != 0 ) {
					inside.emplace_back( thread, seen );
				}
			}
		}
		for( const auto& one : inside ) {
			while( one.first->load() == one.second ) {
				std::this_thread::yield(); // ( a launch is microseconds )
			}
		}
	}

private:
	std::mutex lock;
	std::vector<std::shared_ptr<CEntries>> threads;
};

} // namespace nh
